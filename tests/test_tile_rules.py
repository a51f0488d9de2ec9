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
