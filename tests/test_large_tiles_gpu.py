"""Large tiles (csrc/hip/tile_pipe.h): several groups of row blocks, columns that end inside a lane's eight, and the rule beyond 2,048 rows."""
import pytest
import torch

import test_products_in_tiles_gpu as tiles

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ops = tiles.ops


@pytest.mark.parametrize("tile", range(8, 17))
def test_groups_of_row_blocks(ops, tile):
    """more row blocks than a group of neighbours has (four or eight), the last group not whole; slices and gate and up too"""
    bm, bn = tiles._tiles(ops)[tile]
    M, N, K = 9 * bm + 5, 2 * bn + 20, 320
    x, w = tiles._operands(tile, M, N, K)
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
        tiles._run(ops, x, w, None, out, tile=tile)
        tiles._close(out, x, w, dtype == torch.bfloat16)
    parts = torch.full((2, M, N), float("nan"), device=DEV)
    tiles._run(ops, x, w, parts, out, S=2, tile=tile)
    tiles._close(parts.double().sum(0), x, w, False)
    I = bn + 8
    x, w = tiles._operands(tile + 50, M, 2 * I, K)
    act, gu, want = (torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=DEV) for n in (I, 2 * I, I))
    tiles._run(ops, x, w, None, act, gated=1, act=0, tile=tile, N=I)
    tiles._run(ops, x, w, None, gu, tile=tile)
    ops.swiglu(gu, want)
    # the same roundings of sums that both tiles add in the same order
    assert torch.equal(act, want)


@pytest.mark.parametrize("M,I,K,fused", [(2049, 5632, 2048, True), (9608, 1408, 512, True)])
def test_gated_products_of_many_rows(ops, M, I, K, fused):
    x, w = tiles._operands(M, M, 2 * I, K)
    act = torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
    assert ops.gemm_swiglu(x, w, act) == fused and not ops._tiles_take(M, 2048, K, 1)
    g, u = (x.double() @ w.double().t()).split(I, 1)
    # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each
    assert bool(((act.double() - g * torch.sigmoid(g) * u).abs() <= 4.2 * 2.0 ** -8 * g.abs() * u.abs() + 1e-4).all())


def test_further_tiles(ops, monkeypatch):
    """the tiles that are numbered on from the count: each at its edges, gated, and over several groups of row blocks"""
    import ctypes
    first = ops.lib().kvcm_gemm_tiles_count()

    def size(lib, t):
        rows, cols = ctypes.c_int(), ctypes.c_int()
        assert lib.kvcm_gemm_tiles_size(t, ctypes.byref(rows), ctypes.byref(cols)) == 0
        return rows.value, cols.value
    more = range(first, first + ops.lib().kvcm_gemm_tiles_further())
    assert len(more) == 3
    everything = [size(ops.lib(), t) for t in range(more.stop)]
    assert size_is_refused(ops, more.stop)
    for tile in more:
        with monkeypatch.context() as m:
            m.setattr(tiles, "_tiles", lambda ops, tile=tile: [everything[tile]] * 17)
            run = tiles._run
            m.setattr(tiles, "_run", lambda *a, tile=tile, **kw: run(*a, **{**kw, "tile": tile}))
            tiles.test_every_tile_at_its_edges(ops, 0)
            tiles.test_every_tile_gated(ops, 0)
            test_groups_of_row_blocks(ops, 0)


def size_is_refused(ops, tile):
    import ctypes
    return ops.lib().kvcm_gemm_tiles_size(tile, ctypes.byref(ctypes.c_int()), ctypes.byref(ctypes.c_int())) != 0


@pytest.mark.parametrize("M,I,K", [(49, 8192, 4096), (64, 14336, 4096), (128, 8224, 320), (512, 2048, 192)])
def test_folded_norms_of_many_rows_stay_with_the_tiles_that_take_them(ops, M, I, K):
    x, w = tiles._operands(M + I, M, 2 * I, K)
    ss = torch.rand(M, K // 8, device=DEV) * 8
    rstd = 1.0 / torch.sqrt(ss.double().sum(1, keepdim=True) / K + 1e-5)
    out = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
    rc = ops.lib().kvcm_gemm_skinny_swiglu_normed(x.data_ptr(), w.data_ptr(), ss.data_ptr(), K // 8, 1e-5, out.data_ptr(), M, I, K,
                                                  x.stride(0), w.stride(0), out.stride(0), ops._stream())
    assert rc == 0, ops.lib().kvcm_hip_last_error().decode()
    g, u = (x.double() @ w.double().t() * rstd).split(I, 1)
    # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each; the sums of up to
    # 4,096 products before are off by up to 2 K roundings of 2^-24
    eg, eu = (2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) * rstd).split(I, 1)
    bound = 1.1 * eg * u.abs() + g.abs() * eu + 1.1 * eg * eu
    assert bool(((out.double() - g * torch.sigmoid(g) * u).abs() <= 1.1 * bound + 4.2 * 2.0 ** -8 * (g.abs() * u.abs()) + 1e-5).all())
