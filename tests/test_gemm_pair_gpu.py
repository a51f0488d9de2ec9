"""Two products of at most 8 rows in one launch (``ops.gemm_pair``): every bit of what ``ops.gemm`` computes one after the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF16 = torch.float32, torch.bfloat16


def _product(M, N, K, dtype, seed, pad):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + pad, generator=g, device=DEV).bfloat16()[:, :K]
    w = (torch.randn(N, K + 2 * pad, generator=g, device=DEV) * 0.05).bfloat16()[:, :K]
    return x, w, [torch.full((M, N + pad), 7.0, dtype=dtype, device=DEV)[:, :N] for _ in range(2)]


# one and two row groups, short and long trips in either place, slices of K that are empty or uneven, rows that lie apart
@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("one,two,pad", [((2560, 2048, F32), (8192, 2048, F32), 0), ((128, 4096, BF16), (32, 4096, F32), 0),
                                         ((2048, 2048, F32), (2048, 4096, F32), 8), ((24, 64, BF16), (8, 320, F32), 16),
                                         ((2048, 4160, BF16), (4352, 2112, BF16), 0), ((16, 1024, F32), (4352, 2048, BF16), 8)])
def test_pair(M, one, two, pad):
    from kvcm_amd import ops
    (x1, w1, o1), (x2, w2, o2) = (_product(M, *p, seed=i, pad=pad) for i, p in enumerate((one, two)))
    # (without scratch `gemm` runs none of them in slices; in unsplit form it may not prefer a shape: then the pair is refused)
    takes = [ops._rows8_takes(M, w.shape[0], w.shape[1], o[0].dtype, False) for w, o in ((w1, o1), (w2, o2))]
    assert ops.gemm_pair(x1, w1, o1[0], x2, w2, o2[0], False, False) == all(takes)
    if not all(takes):
        assert (o1[0] == 7).all() and (o2[0] == 7).all()
        return
    for x, w, o in ((x1, w1, o1), (x2, w2, o2)):
        ops.gemm(x, w, o[1], unsplit=True)
        assert torch.equal(o[0], o[1])
        want = x.double() @ w.double().t()
        bound = (x.double().abs() @ w.double().abs().t()) * x.shape[1] * 2.0 ** -24 + (want.abs() * 2.0 ** -8 if o[0].dtype == BF16 else 0)
        assert ((o[0].double() - want).abs() <= bound + 1e-30).all()


def test_pair_refuses():
    from kvcm_amd import ops
    good = _product(4, 64, 1024, F32, 0, 0)
    for M, N, K, dtype in ((9, 64, 1024, F32), (4, 64, 1000, F32), (4, 60, 1024, F32), (4, 64, 1024, BF16)):
        x, w, o = _product(M, N, K, dtype, 1, 0)
        if (M, N, K) == (4, 64, 1024):
            x, o = x[:3], [o[0][:3]]      # not as many rows
        assert not ops.gemm_pair(*good[:2], good[2][0], x, w, o[0])
        assert (good[2][0] == 7).all() and (o[0] == 7).all()
    x, w, o = _product(4, 64, 1024, F32, 1, 0)
    assert not ops.gemm_pair(*good[:2], good[2][0], x.float(), w.float(), o[0])
