"""The rules that pick the tiles of products (csrc/hip/gemm_tiles.hip, moe_grouped.hip), on the host: the sizes their comments name."""
import pytest


@pytest.fixture(scope="module")
def ops():
    from kvcm_amd import ops
    return ops


# (pairs, experts, rows of an expert's matrix, K): the tile that was measured as the fastest, or within a twentieth of it
@pytest.mark.parametrize("n,E,N,K,tiles", [(509, 8, 5632, 2048, {(64, 64), (128, 64)}), (509, 8, 2048, 5632, {(128, 64)}),
                                           (2 * 4072, 8, 2816, 2048, {(256, 256)}), (2 * 8192, 8, 2816, 2048, {(256, 256)}),
                                           (8 * 4072, 64, 512, 256, {(192, 128), (256, 128), (256, 192)}), (2, 64, 512, 256, {(64, 64)})])
def test_tiles_of_routed_experts(ops, n, E, N, K, tiles):
    pick = ops.lib().kvcm_moe_grouped_pick(n, E, N, K)
    assert (pick // 1000, pick % 1000) in tiles


# (M, N, K, gated): products as bench.py's and the command lines' models have them, and others
@pytest.mark.parametrize("M,N,K,gated,here", [(2048, 2560, 2048, 0, 1), (1040, 2048, 2048, 0, 1), (1024, 1024, 512, 0, 1), (2048, 2048, 5632, 0, 1), (513, 2048, 2048, 0, 1),
                                              (2048, 5632, 2048, 1, 1), (1024, 5632, 2048, 1, 1), (32768, 5632, 2048, 1, 1), (8192, 5632, 2048, 1, 1),
                                              (640, 64, 14336, 0, 0), (1040, 8192, 2048, 0, 0), (2048, 8192, 2048, 0, 0), (384, 2048, 5632, 0, 0),
                                              (2048, 256, 5632, 0, 0), (2049, 2560, 2048, 0, 0)])
def test_products_of_many_rows_here_or_by_the_library(ops, M, N, K, gated, here):
    assert ops.lib().kvcm_gemm_tiles_preferred(M, N, K, 1, gated, ops._DT[ops.torch.bfloat16]) == here


# 32-bit results, whose storing costs the library more: us, here / library, launches one after the other
@pytest.mark.parametrize("M,N,K,here", [(2048, 8192, 2048, 1),        # 59.3 / 63.3
                                        (2048, 8256, 2048, 1),        # 75.7 / 90.6
                                        (2048, 2560, 2048, 1),        # 27.0 / 28.3
                                        (4072, 2560, 2048, 0)])
def test_products_with_a_32_bit_result(ops, M, N, K, here):
    assert ops.lib().kvcm_gemm_tiles_preferred(M, N, K, 1, 0, ops._DT[ops.torch.float32]) == here


@pytest.mark.parametrize("M,N,K,S,gated,tile", [(512, 2816, 2048, 1, 1, (128, 96)), (128, 11264, 2048, 2, 0, (128, 96)), (117, 7680, 1600, 4, 0, (128, 128)),
                                                (64, 2048, 2048, 8, 0, (64, 64)), (2048, 2048, 5632, 1, 0, (128, 128)), (32768, 5632, 2048, 1, 1, (256, 256))])
def test_tiles_of_products(ops, M, N, K, S, gated, tile):
    import ctypes
    bm, bn = ctypes.c_int(), ctypes.c_int()
    assert ops.lib().kvcm_gemm_tiles_size(ops.lib().kvcm_gemm_tiles_pick(M, N, K, S, gated), ctypes.byref(bm), ctypes.byref(bn)) == 0
    assert (bm.value, bn.value) == tile
