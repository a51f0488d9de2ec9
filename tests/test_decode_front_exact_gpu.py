"""The attention half in one launch (decode_front.hip) where its products are exact: projections that pick columns leave q, k and v, and the
attention's rows in the stream, without a rounding that an order of sums could move.  So pages are compared bit for bit and the attention entry by entry."""
import math

import numpy as np
import pytest
import torch

from test_decode_front_gpu import _Step
from test_kernels_gpu import DEV, _inv_freq, ops  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


class _Problem:
    """One layer; H = nh hd.  Wqkv's rows pick entries of x, Wo is the identity, the stream is zero: it ends as the attention's bfloat16 rows."""

    def __init__(self, ops, nh, nkv, hd, B, lens, seed, rotate=False, stale=0.0):
        g = torch.Generator().manual_seed(seed)
        self.ops, self.nh, self.nkv, self.hd, self.B, self.lens, self.M, self.H = ops, nh, nkv, hd, B, lens, len(lens), nh * hd
        M, H, W = self.M, self.H, (nh + 2 * nkv) * hd
        self.pick = torch.randint(0, H, (W,), generator=g)
        self.wqkv = torch.zeros(W, H).scatter_(1, self.pick[:, None], 1.0).to(DEV, BF)
        self.wo, self.h = torch.eye(H).to(DEV, BF), torch.randn(M, H, generator=g).bfloat16()
        self.stride = max(-(-c // B) for c in lens) + 1
        pages = M * self.stride + 2
        self.table = torch.randperm(pages - 1, generator=g)[:M * self.stride].reshape(M, self.stride) + 1
        self.k, self.v = torch.randn(M, self.stride * B, nkv, hd, generator=g).bfloat16(), torch.randn(M, self.stride * B, nkv, hd, generator=g).bfloat16()
        for r, c in enumerate(lens):      # what lies behind a row's stored tokens, the place of the newest included
            self.k[r, max(c - 1, 0):] = stale
            self.v[r, max(c - 1, 0):] = stale
        self.pages, self.stale = pages, stale
        self.slots = torch.tensor([int(self.table[r, (c - 1) // B]) * B + (c - 1) % B if c else -1 for r, c in enumerate(lens)], dtype=torch.int32)
        self.angles = None
        if rotate:
            self.angles = torch.empty(M, hd // 2, 2, device=DEV)
            ops.rope_table(torch.tensor([max(c - 1, 0) for c in lens], dtype=torch.int32, device=DEV), torch.tensor(_inv_freq(hd, 1e4), dtype=torch.float32, device=DEV), self.angles)

    def caches(self):
        kc = torch.full((self.pages, self.nkv, self.B, self.hd), self.stale, dtype=BF)
        vc = torch.full((self.pages, self.nkv, self.hd, self.B), self.stale, dtype=BF)
        for r in range(self.M):
            for b in range(self.stride):
                kc[self.table[r, b]] = self.k[r, b * self.B:(b + 1) * self.B].transpose(0, 1)
                vc[self.table[r, b]] = self.v[r, b * self.B:(b + 1) * self.B].permute(1, 2, 0)
        return kc.to(DEV), vc.to(DEV)

    def run(self, one, step=None):
        ops, M, H, nh, nkv, hd = self.ops, self.M, self.H, self.nh, self.nkv, self.hd
        kc, vc = self.caches()
        x, attn, out = torch.zeros(M, H, device=DEV), torch.zeros(M, H, dtype=BF, device=DEV), torch.zeros(M, H, dtype=BF, device=DEV)
        xg, ss = torch.zeros(8, H, dtype=BF, device=DEV), torch.zeros(8, H // 8, device=DEV)
        i32 = lambda t: t.to(DEV, torch.int32).contiguous()
        table, rows, ctx, slots, h = i32(self.table), i32(torch.arange(M)), i32(torch.tensor(self.lens)), i32(self.slots), self.h.to(DEV)
        parts = self.ops.lib().kvcm_decode_front_parts(max(self.lens))

        def attend():
            qkv = ops.gemm(h, self.wqkv, torch.zeros(M, self.wqkv.shape[0], dtype=BF, device=DEV))
            ops.attention_decode_fused(qkv, attn, kc, vc, table, self.stride, rows, ctx, nh, nkv, hd, 1 / math.sqrt(hd), cos_sin=self.angles, slots=slots)

        if one:
            step = step or _Step()
            p = ops.PendingAttention(attend, h, self.wqkv, attn, self.wo, out, None, (kc, vc), table, self.stride, rows, ctx, slots, self.angles, (nh, nkv, hd),
                                     1 / math.sqrt(hd), parts, lambda: ops.decode_front_buffers(step, M, nh, nkv, hd, parts))
            assert p.takes(x, xg, ss)
        else:
            attend()
            p = ops.PendingProduct(attn, self.wo, out)
        ops.gemm_residual_norm(p, x, torch.ones(H, device=DEV, dtype=BF), 1e-5, xg, ss, out)
        torch.cuda.synchronize()
        return x.cpu(), kc.cpu(), vc.cpu(), ss.cpu()

    def exact(self):
        """The attention's rows and the sums of probability times |value|, in 64 bits (no rotation)."""
        nh, nkv, hd = self.nh, self.nkv, self.hd
        qkv = self.h[:, self.pick].double()
        a, b = torch.zeros(self.M, nh, hd, dtype=torch.float64), torch.zeros(self.M, nh, hd, dtype=torch.float64)
        for r, c in enumerate(self.lens):
            if c == 0:
                continue
            k, v = self.k[r, :c].double(), self.v[r, :c].double()
            k[c - 1], v[c - 1] = qkv[r, nh * hd:(nh + nkv) * hd].view(nkv, hd), qkv[r, (nh + nkv) * hd:].view(nkv, hd)
            for head in range(nh):
                kv = head // (nh // nkv)
                p = torch.softmax(k[:, kv] @ qkv[r, head * hd:(head + 1) * hd] / math.sqrt(hd), 0)
                a[r, head], b[r, head] = p @ v[:, kv], p @ v[:, kv].abs()
        return a.view(self.M, -1), b.view(self.M, -1)


def _bits(t):
    return t.view(torch.int16 if t.dtype == BF else torch.int32)


SIZES = [(8, 1, 64, 16, [1, 2, 63, 64, 65, 66, 513, 0]), (4, 2, 64, 8, [1025, 448, 449]), (6, 2, 64, 64, [1537, 700]), (4, 2, 128, 16, [129, 1, 900, 512]),
         (8, 1, 128, 32, [2048]), (2, 2, 128, 24, [600, 25, 24, 23, 100])]


@pytest.mark.parametrize("nh,nkv,hd,B,lens", SIZES)
def test_every_entry_against_64_bits(ops, nh, nkv, hd, B, lens):
    """An entry is off by its rounding to bfloat16 (8 significant bits, half a unit of the last: up to 2^-8 of it) and by the attention's own: probabilities in two
    bfloat16 pieces (2^-16 of each), 32-bit scores (64 or 128 products of up to about 20 in all: an exponent off by 1e-4 at the worst) and sums,
    together less than 2^-12 of the sum of probability times |value|.  Pages hold exactly what was picked."""
    p = _Problem(ops, nh, nkv, hd, B, lens, seed=nh + hd + len(lens))
    x, kc, vc, ss = p.run(True)
    want, size = p.exact()
    off = (x.double() - want).abs()
    bound = 2 ** -8 * want.abs() + 2 ** -12 * size
    assert bool((off <= bound).all()), float((off / bound.clamp_min(1e-30)).max())
    assert torch.allclose(ss[:p.M].sum(1), (x * x).sum(1), rtol=1e-5)
    x3, kc3, vc3, _ = p.run(False)
    assert torch.equal(_bits(kc), _bits(kc3)) and torch.equal(_bits(vc), _bits(vc3))
    assert bool(((x - x3).abs() <= 2 ** -7 * x3.abs() + 2 ** -12 * size).all())      # (neighbours where their sums lie about a middle)


@pytest.mark.parametrize("nh,nkv,hd,B,lens", SIZES)
@pytest.mark.parametrize("stale", (float("nan"), float("inf"), -3e38))
def test_what_lies_behind_a_context_is_nothing(ops, nh, nkv, hd, B, lens, stale):
    """Rotated keys, and pages full of anything behind each row's tokens: every bit as with zeros there, pages as of three launches."""
    clean, full = (_Problem(ops, nh, nkv, hd, B, lens, seed=3, rotate=True, stale=s) for s in (0.0, stale))
    got, want, three = full.run(True), clean.run(True), full.run(False)
    assert torch.isfinite(got[0]).all() and torch.equal(_bits(got[0]), _bits(want[0]))
    assert torch.equal(_bits(got[1]), _bits(three[1])) and torch.equal(_bits(got[2]), _bits(three[2]))


@pytest.mark.parametrize("where", ("old value", "new value", "old key", "query"))
def test_values_that_are_not_finite(ops, where):
    """They reach the rows that they reach in three launches (all of a row, through the output product), and no others."""
    p = _Problem(ops, 4, 2, 64, 16, [700, 65, 30], seed=11)
    if where == "old value":
        p.v[0, 13, 1, 5], p.v[1, 64 - 2, 0, 3] = float("inf"), float("nan")
    elif where == "old key":
        p.k[0, 640, 1, 5] = float("nan")
    else:      # an entry of x that only this place picks
        at = {"new value": (4 + 2 + 1) * 64 + 7, "query": 64 + 9}[where]
        p.pick[p.pick == 17] = 18
        p.pick[at] = 17
        p.wqkv = torch.zeros(p.wqkv.shape).scatter_(1, p.pick[:, None], 1.0).to(DEV, BF)
        p.wqkv[:, 17] = 0
        p.wqkv[at, 17] = 1.0
        p.h[0, 17], p.h[1, 17] = 3e38, 0.0      # finite in the product with zeros; scores with it are not
        p.h[2, 17] = 0.0
    got, three = p.run(True)[0], p.run(False)[0]
    both = torch.isfinite(got).all(1)
    assert both.tolist() == torch.isfinite(three).all(1).tolist() and bool(both[2])
    assert bool(both[0]) == (where in ("new value", "old key"))      # (3e38 as a value is a large result; a score that is no number has no share)
    assert bool(((got - three)[both].abs() <= 2 ** -7 * three[both].abs() + 2 ** -10).all())      # (a rounding to bfloat16; the sum of probability times |other value| is below 4)


def test_layers_of_other_layouts_share_the_buffers(ops):
    """One step whose layers change between head layouts, the second of which needs more room than the first left: as each on its own."""
    a, b = _Problem(ops, 4, 2, 64, 16, [70, 600, 3], seed=1), _Problem(ops, 8, 2, 128, 16, [1100, 5, 64], seed=2)
    want = {id(p): p.run(True) for p in (a, b)}
    step = _Step()
    for p in (a, b, a, a, b, b, a):
        assert all(torch.equal(_bits(g), _bits(w)) for g, w in zip(p.run(True, step), want[id(p)]))


def test_decode_steps_of_an_engine_take_it(ops, tmp_path, monkeypatch):
    """Recorded decode steps run one such launch a layer up to 8 rows and contexts of 2,048, none otherwise."""
    from kvcm_amd import Engine, EngineConfig
    from kvcm_amd.config.model_config import LlamaConfig
    from kvcm_amd.weights.random_init import write_model_dir
    raw = dict(vocab_size=128, hidden_size=128, intermediate_size=192, num_hidden_layers=3, num_attention_heads=2, num_key_value_heads=1, head_dim=64,
               max_position_embeddings=4096, rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)
    d = str(tmp_path / "m")
    write_model_dir(d, "LlamaForCausalLM", LlamaConfig.from_dict(raw), seed=0, dtype=BF)
    calls, call = [], ops._call

    def counting(name, *args):
        calls.append(name)
        return call(name, *args)

    monkeypatch.setattr(ops, "_call", counting)
    for prompts, layers in (([5], 3), ([5, 7, 900, 30, 1, 2, 3, 4], 3), ([1500, 20], 3), ([3] * 9, 0), ([2100], 0)):
        eng = Engine(d, EngineConfig(dtype="bfloat16", block_size=16, num_blocks=512, max_seq_len=4096, max_num_seqs=16, max_batched_tokens=4096))
        per_step, last = [], eng.decode_graphs.record

        def record(sampling):
            calls.clear()
            out = last(sampling)
            per_step.append((eng.decode_graphs.shape.max_run, calls.count("kvcm_decode_front")))
            return out

        eng.decode_graphs.record = record
        eng.generate([np.arange(n).__mod__(128).tolist() for n in prompts], 3)
        decodes = [n for run, n in per_step if run == 1]
        assert decodes and all(n == layers for n in decodes), (prompts, per_step)
