"""32-bit products (csrc/hip/gemm_f32.hip): the kernels that share one sequence of operations per element, at the edges of what each takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from kvcm_amd import ops as _ops
    _ops.lib()
    return _ops


def _product(ops, x, w, ldy=0):
    M, N = x.shape[0], w.shape[0]
    room = torch.full((M, N + ldy), float("nan"), device=DEV)
    ops.gemm(x, w, room[:, :N])
    assert torch.isnan(room[:, N:]).all()
    return room[:, :N]


# K of one segment, of fewer segments than waves, of segments of unequal lengths, ragged K, K of whole units and of one unit more
@pytest.mark.parametrize("K", [257, 288, 300, 320, 511, 512, 1056, 2048, 2079])
@pytest.mark.parametrize("N", [1, 7, 8, 65, 520])
def test_rows_in_blocks_of_eight_columns_give_the_tiles_bits(ops, N, K):
    g = torch.Generator(device=DEV).manual_seed(N * K)
    # (tiles: many rows; rows that begin at any float; values that are not finite stay with their rows and columns)
    x = torch.randn(2000, K + 3, generator=g, device=DEV)[:, 1:K + 1]
    w = torch.randn(N, K + 1, generator=g, device=DEV)[:, :K]
    full = _product(ops, x, w)
    bound = 2.0 * K * 2.0 ** -24 * (x[:64].abs().double() @ w.abs().double().t())
    assert bool(((full[:64].double() - x[:64].double() @ w.double().t()).abs() <= bound).all())
    for M in (1, 2, 3, 7, 8, 9):
        assert torch.equal(_product(ops, x[5:5 + M], w, 3), full[5:5 + M]), M
        assert torch.equal(_product(ops, x[5:5 + M].contiguous(), w.contiguous()), full[5:5 + M]), M
    x[6, K // 2], w[N - 1, K - 1] = float("nan"), float("inf")
    got = _product(ops, x[5:10], w)
    keep = [0, 2, 3, 4]
    assert torch.equal(got[keep, :N - 1], full[5:10][keep, :N - 1]) and torch.isnan(got[1]).all() and not torch.isfinite(got[:, N - 1]).any()


@pytest.mark.parametrize("M,N,K", [(65, 7400, 288), (64, 7400, 320), (300, 2080, 1056), (1500, 1999, 512), (700, 4100, 416), (32, 30720, 512), (20, 16100, 320)])
def test_tiles_through_the_ring_give_the_staged_tiles_bits(ops, M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    wide = torch.randn(M, K + 3, generator=g, device=DEV)
    x, w = wide[:, 1:K + 1], torch.randn(N, K, generator=g, device=DEV)      # (rows that begin at any float are staged through registers)
    staged, ringed = _product(ops, x, w, 1), _product(ops, x.contiguous(), w, 1)
    assert torch.equal(staged, ringed)
    bound = 2.0 * K * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t())
    assert bool(((ringed.double() - x.double() @ w.double().t()).abs() <= bound).all())
