"""The attention half of a decoding layer in one launch (decode_front.hip) against the three launches it stands for: QKV product,
attention from the projection, output product with the folded norm."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, _inv_freq, _np, _paged_problem, _t, _vt, ops  # noqa: F401

pytestmark = pytest.mark.gpu


class _Step:
    def __init__(self):
        self.shared, self.held = {}, {}

    def flat(self, name, numel, dtype):
        if name not in self.held or self.held[name].numel() < numel:
            self.held[name] = torch.randint(-2 ** 31, 2 ** 31 - 1, (numel,), device=DEV, dtype=dtype)      # whatever lies there is emptied first
        return self.held[name]


def _layers(ops, H, nh, nkv, hd, B, lens, layers, seed, rotate=True, stored=None, scaled_first=False):
    """-> a function that runs `layers` attention halves on fresh copies, one launch or three, and gives stream, xg, ss and caches."""
    rng = np.random.default_rng(seed)
    P = _paged_problem(rng, [max(c, 1) for c in lens], nh, nkv, hd, B, all_rows=False)
    M, W = len(lens), (nh + 2 * nkv) * hd
    order = rng.permutation(M)                      # rows are not in the order of their sequences
    ctx = np.asarray(lens, np.int32)[order]
    pos = np.maximum(ctx - 1, 0)
    slots = np.array([P["tables"][s, p // B] * B + p % B if c > 0 else -1 for s, p, c in zip(order, pos, ctx)], np.int32)
    if stored is not None:
        slots[~np.asarray(stored)[order]] = -1
    tables, row_seq, ctx_t, slots_t = (_t(v, torch.int32) for v in (P["tables"], order, ctx, slots))
    table = None
    if rotate:
        table = torch.empty(M, hd // 2, 2, device=DEV)
        ops.rope_table(_t(pos, torch.int32), _t(_inv_freq(hd, 1e4), torch.float32), table)
    bf = torch.bfloat16
    wqkv = [_t(rng.normal(size=(W, H)) / math.sqrt(H), bf) for _ in range(layers)]
    wo = [_t(rng.normal(size=(H, nh * hd)) / math.sqrt(nh * hd), bf) for _ in range(layers)]
    g = [_t(1 + 0.1 * rng.normal(size=H), bf) for _ in range(layers)]
    x0 = _t(rng.normal(size=(M, H)), torch.float32)
    normed = torch.empty(M, H, dtype=bf, device=DEV)
    ops.rmsnorm(x0, g[0], normed, 1e-5)

    def run(one_launch, polls=-1):
        x = x0.clone()
        kc, vc = _t(P["Kc"], bf), _vt(P["Vc"], bf)
        pairs = [(torch.zeros(8, H, dtype=bf, device=DEV), torch.zeros(8, H // 8, device=DEV)) for _ in range(2)]
        h, step = normed, _Step()
        if scaled_first:                            # a product of nothing leaves the norm's first half
            zero = ops.PendingProduct(torch.zeros(M, 64, dtype=bf, device=DEV), torch.zeros(H, 64, dtype=bf, device=DEV), torch.zeros(M, H, dtype=bf, device=DEV))
            h = ops.gemm_residual_norm(zero, x, g[0], 1e-5, *pairs[1], normed)
        for i in range(layers):
            attn = torch.zeros(M, nh * hd, dtype=bf, device=DEV)
            out = torch.zeros(M, H, dtype=bf, device=DEV)
            parts = ops.decode_front_parts(M, H, nh, nkv, hd, B, max(lens))
            assert parts == -(-max(lens) // 512)

            def attend(i=i, h=h, attn=attn):
                qkv = ops.gemm(h, wqkv[i], torch.zeros(M, W, dtype=bf, device=DEV))
                ops.attention_decode_fused(qkv, attn, kc, vc, tables, P["max_blocks"], row_seq, ctx_t, nh, nkv, hd, 1 / math.sqrt(hd), cos_sin=table, slots=slots_t)

            product = ops.PendingAttention(attend, h, wqkv[i], attn, wo[i], out, None, (kc, vc), tables, P["max_blocks"], row_seq, ctx_t, slots_t, table,
                                           (nh, nkv, hd), 1 / math.sqrt(hd), parts, lambda: ops.decode_front_buffers(step, M, nh, nkv, hd, parts))
            product.polls = polls
            if not one_launch:
                attend()
                product = ops.PendingProduct(attn, wo[i], out)
            else:
                assert product.takes(x, *pairs[i % 2])
            h = ops.gemm_residual_norm(product, x, g[i], 1e-5, *pairs[i % 2], normed.clone())
        torch.cuda.synchronize()
        return _np(x), _np(h.xg), _np(h.ss), _np(kc), _np(vc)

    return run, _np(x0), slots


@pytest.mark.parametrize("H,nh,nkv,hd,B,lens", [
    (2048, 32, 4, 64, 16, [600]),
    (2048, 32, 4, 64, 16, [513, 1, 2, 63, 64, 65, 66, 0]),
    (2048, 32, 4, 64, 16, [1024, 129, 1023]),
    (2048, 32, 4, 64, 16, [2048, 0, 1025, 1537, 128, 257, 512, 2]),
    (320, 5, 1, 64, 8, [449, 450, 448, 511]),
    (64, 2, 2, 64, 24, [100, 23, 24, 25, 26]),
    (192, 6, 2, 64, 64, [1500, 64]),
    (4096, 32, 8, 128, 16, [777, 3]),
    (256, 7, 1, 128, 32, [1, 0, 640, 32, 33]),
    (128, 8, 8, 128, 16, [1100]),
])
def test_attention_half_in_one_launch(ops, H, nh, nkv, hd, B, lens):
    """Every edge of a window, of a part and of a page, a row's first token, padding rows, rows in another order than their sequences,
    K slices of unequal length, three layers through the two buffers in turn.  What differs is the order of 32-bit sums, that
    is single bfloat16 roundings: of q, k and v, of the attention's rows, of the product (at most a unit of the last place, 2^-7 of
    their size, most of them equal).  Entry by entry: test_decode_front_exact_gpu.py."""
    run, x0, slots = _layers(ops, H, nh, nkv, hd, B, lens, 3, seed=H + nh + len(lens), scaled_first=len(lens) % 2 == 0)
    want, got = run(False), run(True)
    live = np.array([s >= 0 for s in slots])
    for a, b in zip(got, want):
        assert np.isfinite(a).all()
    assert np.linalg.norm(got[0][live] - want[0][live]) <= 2 ** -7 * np.linalg.norm(want[0][live] - x0[live])
    assert np.linalg.norm(got[1][live] - want[1][live]) <= 2 ** -7 * np.linalg.norm(want[1][live])
    np.testing.assert_allclose(got[2][live].sum(-1), (got[0][live] ** 2).sum(-1), rtol=1e-5)
    for a, b in ((got[3], want[3]), (got[4], want[4])):      # the same places of the caches, to the last rounding or two of later layers
        assert np.abs(a - b).max() <= 2 ** -5 * max(1.0, np.abs(b).max()) and (a != b).mean() <= 0.25 * (want[3] != 0).mean()
    again = run(True)
    assert all(np.array_equal(a, b) for a, b in zip(got, again))


def test_attention_half_in_one_launch_without_rotation_and_without_storing(ops):
    """No table of angles; rows whose key is in the cache already (nothing is stored, the context is read as it is)."""
    run, x0, slots = _layers(ops, 256, 8, 2, 64, 16, [300, 64, 65, 1], 2, seed=5, rotate=False, stored=[True, False, False, False])
    want, got = run(False), run(True)
    assert np.linalg.norm(got[0] - want[0]) <= 2 ** -7 * np.linalg.norm(want[0] - x0)
    assert np.abs(got[3] - want[3]).max() <= 2 ** -5 * np.abs(want[3]).max()


def test_attention_half_refusals(ops):
    lib = ops.lib()
    assert ops.decode_front_parts(8, 2048, 32, 4, 64, 16, 2048) == 4 and ops.decode_front_parts(8, 2048, 32, 4, 64, 16, 2049) == 0
    for shape in ((9, 2048, 32, 4, 64, 16), (0, 2048, 32, 4, 64, 16), (4, 2040, 32, 4, 64, 16), (4, 2048, 36, 4, 64, 16), (4, 2048, 32, 4, 96, 16),
                  (4, 2048, 32, 4, 64, 12), (4, 2048, 30, 4, 64, 16)):
        assert ops.decode_front_parts(*shape, 512) == 0
    words = lib.kvcm_decode_front_words(8, 32, 4, 64, 2)
    assert words == 8 * (2560 + 1024 + 32 * 66) and words % 4 == 0
    with pytest.raises(ops.KernelError, match="too small"):
        ops._call("kvcm_decode_front", *([1 << 20, 2048] * 2), 0, 0, 0.0, 1 << 20, 2048, 8, 2048, 0, *([1 << 20] * 4), 64, 8, *([1 << 20] * 2), 32, 4, 64, 16, 0.1,
                  1 << 20, 1 << 20, 1, 2 << 20, 1 << 20, 1 << 20, 2 << 20, words - 4, 2, ops._stream())
