"""Steps in which every sequence runs one row: convolution, rotation, page write, attention and pooled entry in one launch
(``attention_window_pool_rows``) against the launches one by one, which have references of their own: every bit of the output, the pages, the
convolution's state and the pooled entries is the same."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

CONV = [dict(nh=32, nkv=4, d=64, dv=64, B=16, W=512, P=64, taps=4, rot=64, top=1300),      # one chunk a wave, pooled chunks besides
        dict(nh=8, nkv=2, d=64, dv=64, B=16, W=96, P=2, taps=4, rot=32, top=2300),         # several pooled chunks a wave
        dict(nh=4, nkv=2, d=24, dv=40, B=8, W=16, P=4, taps=1, rot=0, top=70),             # sizes that are no tile's, no state
        dict(nh=32, nkv=2, d=16, dv=8, B=24, W=70, P=16, taps=8, rot=16, top=900),         # sixteen heads, most taps; pages and blocks out of step
        dict(nh=4, nkv=1, d=64, dv=64, B=8, W=0, P=0, taps=3, rot=64, top=900)]            # every token, more chunks than waves


def _setup(s, seed):
    g = torch.Generator().manual_seed(seed)
    nh, nkv, d, dv, B, W, P = s["nh"], s["nkv"], s["d"], s["dv"], s["B"], s["W"], s.get("P", 0)
    ctx = sorted({1, 2, 5, B, B + 1, 63, 64, 65, s["top"], s["top"] - s["top"] % max(P, 2)} | ({W, W + 1, W + max(P, 1)} if W else set()))
    ctx = [min(c, s["top"]) for c in ctx] + [0, 7]      # a padding row, and one whose key is not stored
    T, stride = len(ctx), -(-s["top"] // B)
    pages = T * stride + 1
    order = torch.randperm(pages - 1, generator=g)[:T * stride].reshape(T, stride)
    rand = lambda *n: torch.randn(*n, generator=g)
    kc, vc = rand(pages, nkv, B, d).bfloat16(), rand(pages, nkv, dv, B).bfloat16()
    slots = [-1] * T
    for i, c in enumerate(ctx):
        if c and i < T - 1:
            slots[i] = int(order[i][(c - 1) // B]) * B + (c - 1) % B
        for t in range(max(0, c - (i < T - 1)), stride * B):      # what no token wrote may hold anything
            kc[order[i][t // B], :, t % B] = float("nan")
            vc[order[i][t // B], :, :, t % B] = float("nan")
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).to(DEV)
    pos = [max(c - 1, 0) for c in ctx]
    step = SimpleNamespace(rows=T, seqs=T, max_run=1, row_seq=i32(range(T)), positions=i32(pos), ctx_lens=i32(ctx), run_start=i32(range(T + 1)),
                           seq_start=i32(pos), seq_end=i32(ctx), state_slots=i32([v if i != 1 else -1 for i, v in enumerate(torch.randperm(T, generator=g).tolist())]))
    E = -(-B // P) if P else 0
    pk, pv = (rand(pages, nkv, E, n).to(DEV) if P else None for n in (d, dv))
    C = (nh + nkv) * d + nkv * dv
    proj = rand(T, C + 8).to(DEV)[:, :C]
    angle = rand(T, max(s["rot"] // 2, 1)) * 3
    cos_sin = torch.stack([angle.cos(), angle.sin()], -1).contiguous().to(DEV) if s["rot"] else None
    return SimpleNamespace(step=step, kc=kc.to(DEV), vc=vc.to(DEV), pk=pk, pv=pv, table=order.to(torch.int32).contiguous().to(DEV), stride=stride,
                           slots=i32(slots), proj=proj, cos_sin=cos_sin, C=C, T=T, rand=lambda *n: rand(*n).to(DEV))


def _same(a, b, what):
    view = torch.int16 if a.dtype == torch.bfloat16 else torch.int32
    assert torch.equal(a.view(view), b.view(view)), what


@pytest.mark.parametrize("s", CONV, ids=lambda s: "%d-%d-%d" % (s["nh"], s["d"], s["taps"]))
def test_convolution_to_attention(s):
    from kvcm_amd import ops
    x = _setup(s, s["nh"] + s["d"])
    nh, nkv, d, dv, P, T, st = s["nh"], s["nkv"], s["d"], s["dv"], s["P"], x.T, x.step
    assert ops.attention_window_pool_rows_supported(nh, nkv, d, dv, torch.bfloat16, s["B"])
    conv, bias, temp = x.rand(x.C, s["taps"]), x.rand(x.C), 1 + x.rand(nh).abs()
    state = x.rand(T, s["taps"] - 1, x.C) if s["taps"] > 1 else None
    results = []
    for one in (False, True):
        kc, vc = x.kc.clone(), x.vc.clone()
        pk, pv = (t.clone() if P else None for t in (x.pk, x.pv))
        cs = state.clone() if state is not None else None
        out = torch.full((T, nh * dv + 8), 7.0, dtype=torch.bfloat16, device=DEV)[:, :nh * dv]
        if one:
            ops.attention_window_pool_rows(x.proj, out, kc, vc, pk, pv, st, x.table, x.stride, x.slots, nh, nkv, d, dv, d ** -0.5, s["W"], P, conv, cs,
                                           conv_bias=bias, head_scale=temp, cos_sin=x.cos_sin, rot=s["rot"])
        else:
            mixed, q = torch.empty(T, x.C, device=DEV), torch.empty(T, nh * d, dtype=torch.bfloat16, device=DEV)
            ops.short_conv(x.proj, conv, mixed, st, cs, bias_in=bias, update_state=True)
            ops.rotate_store(mixed, q, nh, nkv, d, dv, cos_sin=x.cos_sin, rot=s["rot"], slots=x.slots, kcache=kc, vcache=vc, rows=T)
            if P:
                ops.pool_update(kc, vc, pk, pv, x.table, x.stride, st.row_seq, st.positions, x.slots, nkv, d, dv, P, T)
            ops.attention_window_pool(q, out, kc, vc, pk, pv, x.table, x.stride, st.row_seq, st.ctx_lens, nh, nkv, d, dv, d ** -0.5, s["W"], P,
                                      head_scale=temp, rows=T)
        results.append([t for t in (out, kc, vc, pk, pv, cs) if t is not None])
    assert torch.isfinite(results[0][0].float()).all()
    for a, b in zip(*results):
        _same(a.contiguous(), b.contiguous(), tuple(a.shape))


def test_what_it_refuses():
    from kvcm_amd import ops
    sup = ops.attention_window_pool_rows_supported
    for nh, nkv, d, dv, B in ((4, 4, 64, 64, 16), (34, 2, 64, 64, 16), (8, 2, 68, 64, 16), (8, 2, 72, 64, 16), (8, 2, 64, 72, 16), (8, 2, 64, 64, 12)):
        assert not sup(nh, nkv, d, dv, torch.bfloat16, B)
    assert not sup(8, 2, 64, 64, torch.float32, 16)


def test_it_is_left_alone_where_workgroups_outnumber_the_chip():
    """256 workgroups have a CU each; more rows ran up to 1.8 times as long as in the launches one by one."""
    from kvcm_amd import ops
    takes = ops.attention_window_pool_rows_takes
    for nkv, most in ((4, 64), (8, 32), (3, 85), (1, 256)):
        assert takes(most, 4 * nkv, nkv, 64, 64, torch.bfloat16, 16) and not takes(most + 1, 4 * nkv, nkv, 64, 64, torch.bfloat16, 16)
    assert not takes(0, 8, 2, 64, 64, torch.bfloat16, 16) and not takes(1, 8, 512, 64, 64, torch.bfloat16, 16)
    assert not takes(8, 8, 2, 64, 64, torch.float32, 16) and not takes(8, 8, 2, 72, 64, torch.bfloat16, 16)
