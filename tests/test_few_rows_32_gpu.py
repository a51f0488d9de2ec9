"""32-bit decode rows: products with the norm in front and SwiGLU or the residual addition behind (gemm_f32_few.hip), rotation, page write
and attention in one launch (attention_generic.hip).  All have the bits of the launches they stand for."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, _inv_freq, _paged_problem, _t, _vt, ops  # noqa: F401

pytestmark = pytest.mark.gpu


def _rand(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


# the edges of the three sizes of registers and of a unit
@pytest.mark.parametrize("K", [4, 28, 64, 68, 96, 128, 132, 176, 252, 256])
@pytest.mark.parametrize("N", [1, 4, 15, 33, 64, 130, 2048])
def test_norm_in_front_and_swiglu_or_addition_behind_keep_the_bits(ops, N, K):
    g = torch.Generator(device=DEV).manual_seed(N * K)
    w, gu, weight = _rand(g, N, K), _rand(g, 2 * N, K), 1 + 0.1 * _rand(g, K)
    wide = _rand(g, 64, K + 5)
    for M in (1, 2, 5, 8, 15, 16, 17, 64):
        x = wide[:M, :K].clone(memory_format=torch.contiguous_format)
        assert ops.f32_few_takes(M, K)
        # addition behind; rows of X that begin at any float
        for rows in (x, wide[:M, 3:K + 3]):
            want = ops.gemm(rows, w, torch.empty(M, N, device=DEV))
            stream = _rand(g, M, N)
            total = stream.clone()
            ops.add_residual(total, want)
            room = torch.full((M + 1, N), 7.0, device=DEV)
            room[:M] = stream
            ops.gemm_residual(ops.PendingProduct(rows, w, want), room[:M])
            assert torch.equal(room[:M], total) and bool((room[M] == 7.0).all())
        both = ops.gemm(x, gu, torch.empty(M, 2 * N, device=DEV))
        act, normed = torch.empty(M, N, device=DEV), torch.empty_like(x)
        ops.swiglu(both, act)
        got = torch.full((M, N + 1), float("nan"), device=DEV)
        assert ops.gemm_swiglu(x, gu, got[:, :N]) and torch.equal(got[:, :N], act) and bool(got[:, N].isnan().all())
        assert ops.can_norm_rows(x, weight, normed)
        ops.rmsnorm(x, weight, normed, 1e-5)
        h = ops.RowsToNorm(x, weight, 1e-5, torch.empty_like(x))
        want, got = ops.gemm(normed, w, torch.empty(M, N, device=DEV)), torch.full((M, N + 1), float("nan"), device=DEV)
        assert torch.equal(ops.gemm(h, w, got[:, :N]), want) and bool(got[:, N].isnan().all())
        ops.swiglu(ops.gemm(normed, gu, both), act)
        assert ops.gemm_swiglu(h, gu, got[:, :N]) and torch.equal(got[:, :N], act)
        assert torch.equal(h.materialize(), normed)


# segments: one unit more than one chain takes, unequal lengths, the widest rows
@pytest.mark.parametrize("K", [260, 288, 1028, 2048, 8192])
@pytest.mark.parametrize("I", [1, 3, 4, 130, 1025])
def test_swiglu_behind_wider_rows_keeps_the_bits(ops, I, K):
    g = torch.Generator(device=DEV).manual_seed(I * K)
    gu, wide = _rand(g, 2 * I, K + 1)[:, :K], _rand(g, 8, K + 5)
    for M in (1, 2, 3, 7, 8):
        for x in (wide[:M, :K].clone(memory_format=torch.contiguous_format), wide[:M, 3:K + 3]):
            act, got = torch.empty(M, I, device=DEV), torch.full((M, I + 1), float("nan"), device=DEV)
            ops.swiglu(ops.gemm(x, gu, torch.empty(M, 2 * I, device=DEV)), act)
            assert ops.gemm_swiglu(x, gu, got[:, :I]) and torch.equal(got[:, :I], act) and bool(got[:, I].isnan().all())
    x[0, K // 2] = float("inf")
    assert ops.gemm_swiglu(x, gu, got[:, :I]) and torch.equal(got[1:, :I], act[1:]) and not bool(torch.isfinite(got[0]).any())


def test_values_that_are_not_finite_stay_with_their_rows(ops):
    g = torch.Generator(device=DEV).manual_seed(1)
    for K in (64, 200):
        x, w, weight = _rand(g, 5, K), _rand(g, 40, K), 1 + 0.1 * _rand(g, K)
        plain = ops.gemm(ops.RowsToNorm(x, weight, 1e-5, x), w, torch.empty(5, 40, device=DEV)).clone()
        x[1, K // 2], x[3, 0] = float("nan"), float("inf")
        got = ops.gemm(ops.RowsToNorm(x, weight, 1e-5, x), w, torch.empty(5, 40, device=DEV))
        assert torch.equal(got[[0, 2, 4]], plain[[0, 2, 4]]) and bool(got[[1, 3]].isnan().all())


def test_few_rows_refusals(ops):
    for M, K, takes in ((64, 256, 1), (65, 256, 0), (8, 260, 0), (1, 30, 0), (0, 64, 0)):
        assert ops.f32_few_takes(M, K) == bool(takes), (M, K)
    for M, I, K, takes in ((8, 5632, 2048, 1), (9, 5632, 2048, 0), (1, 5632, 256, 0), (2, 14336, 4096, 1), (3, 14336, 4096, 0), (1, 16000, 2048, 0), (1, 64, 8196, 0), (1, 64, 510, 0)):
        assert ops.lib().kvcm_gemm_f32_swiglu_preferred(M, I, K) == takes, (M, I, K)
    x = torch.zeros(9, 512, device=DEV)
    with pytest.raises(ops.KernelError, match="unsupported shape"):
        ops.gemm_residual(ops.PendingProduct(x, torch.zeros(8, 512, device=DEV), x), torch.zeros(9, 8, device=DEV))
    assert not ops.gemm_swiglu(x, torch.zeros(16, 512, device=DEV), torch.zeros(9, 8, device=DEV))


@pytest.mark.parametrize("nh,nkv,hd,B,window", [(4, 2, 16, 16, 0), (16, 1, 16, 4, 0), (3, 1, 32, 16, 0), (32, 4, 64, 16, 0), (8, 8, 64, 24, 40), (6, 2, 128, 16, 0)])
@pytest.mark.parametrize("rotate", [True, False])
def test_rotation_page_write_and_attention_in_one_launch_keep_the_bits(ops, nh, nkv, hd, B, window, rotate):
    rng = np.random.default_rng(nh + hd)
    for lens in ([1], [65, 1, 64, 0, 63], [17, 300, 5, 129, 64, 1, 16, 1025]):
        P = _paged_problem(rng, [max(c, 1) for c in lens], nh, nkv, hd, B, all_rows=False)
        M = len(lens)
        order = rng.permutation(M)
        ctx = np.asarray(lens, np.int32)[order]
        pos = np.maximum(ctx - 1, 0)
        slots = np.array([P["tables"][s, p // B] * B + p % B if c > 0 else -1 for s, p, c in zip(order, pos, ctx)], np.int32)
        slots[0] = -1                                   # (a row whose key is in its page already)
        tables, seq, ctx_t, slots_t = (_t(v, torch.int32) for v in (P["tables"], order, ctx, slots))
        rows = _t(rng.normal(size=(M, (nh + 2 * nkv) * hd)), torch.float32)
        table = torch.empty(M, hd // 2, 2, device=DEV)
        ops.rope_table(_t(pos, torch.int32), _t(_inv_freq(hd, 1e4), torch.float32), table)
        table = table if rotate else None
        kc, vc = _t(P["Kc"], torch.float32), _vt(P["Vc"], torch.float32)
        kc2, vc2, given = kc.clone(), vc.clone(), rows.clone()
        want, got = torch.zeros(M, nh * hd, device=DEV), torch.full((M, nh * hd), 5.0, device=DEV)
        ops.attention_f32_decode(rows, got, kc2, vc2, tables, P["max_blocks"], seq, ctx_t, nh, nkv, hd, 1 / math.sqrt(hd), slots_t, cos_sin=table, window=window)
        assert torch.equal(rows, given)
        ops.rope_cache(rows, nh, nkv, hd, slots=slots_t, kcache=kc, vcache=vc, block_size=B, cos_sin=table)
        ops.attention(rows, want, kc, vc, tables, P["max_blocks"], seq, ctx_t, nh, nkv, hd, 1 / math.sqrt(hd), window)
        assert torch.equal(kc, kc2) and torch.equal(vc, vc2) and torch.equal(got, want)
    assert not ops.attention_f32_decode_supported(4, 2, 48, 16) and not ops.attention_f32_decode_supported(32, 1, 64, 16)
