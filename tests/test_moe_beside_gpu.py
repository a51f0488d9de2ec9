"""A shared feed-forward (and a route by a table) in the experts' two launches (``ops.moe_few_beside``) against 64 bits: the activations from the operands,
the output from the activations as stored.  Bounds: 2^-24 per 32-bit operation of a sum, times the sum of the terms' sizes; 2^-8 for what is stored."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda", torch.bfloat16


def _sum_bound(a, b):
    return (a.abs() @ b.abs().transpose(-1, -2)) * (a.shape[-1] + 2) * 2.0 ** -24


def _act_check(act, x, gate, up, scale):
    z0, z1 = (x @ gate.t()) * scale, (x @ up.t()) * scale
    e0, e1 = _sum_bound(x, gate) * scale, _sum_bound(x, up) * scale
    want = z0 * torch.sigmoid(z0) * z1
    bound = want.abs() * (2.0 ** -8 + 2.0 ** -18) + 1.2 * e0 * (z1.abs() + e1) + (z0.abs() + e0) * e1 + 1e-30      # silu's slope is below 1.1
    assert ((act.double() - want).abs() <= bound).all()


# (rows, width in, columns an expert, width out, slots, experts, shared columns, by table, weights on the input)
@pytest.mark.parametrize("T,K,F,H,top,E,Fs,table,weigh_input",
                         [(1, 2048, 1408, 2048, 2, 8, 2816, True, False), (8, 2048, 1408, 2048, 2, 8, 2816, True, False),
                          (16, 256, 64, 128, 4, 32, 64, True, True), (3, 192, 128, 64, 1, 3, 832, False, False), (8, 1024, 704, 1024, 2, 8, 1408, False, True),
                          (20, 128, 64, 72, 3, 5, 320, False, False), (64, 64, 64, 8, 1, 2, 128, True, False), (9, 320, 192, 136, 2, 4, 64, True, False)])
def test_beside(T, K, F, H, top, E, Fs, table, weigh_input):
    from kvcm_amd import ops
    from kvcm_amd.parts.routed_parts import interleave_gate_up
    g = torch.Generator(device=DEV).manual_seed(T + K + F)
    rand = lambda *n, by=1.0: (torch.randn(*n, generator=g, device=DEV) * by).to(BF16)
    h = rand(T, K + 8)[:, :K]
    gate, up, down = rand(E, F, K, by=K ** -0.5), rand(E, F, K, by=K ** -0.5), rand(E, H, F, by=F ** -0.5)
    s_up, s_down = rand(2 * Fs, K, by=K ** -0.5), rand(H, Fs, by=Fs ** -0.5)
    w_up = interleave_gate_up(gate, up).contiguous()
    vocab = 37
    tab = torch.stack([torch.randperm(max(E, top), generator=g, device=DEV)[:top] for _ in range(vocab)]).to(torch.int32)
    tab = torch.cat([tab, tab], 1)[:, :top] if top == 1 else torch.cat([tab, tab], 1)      # (rows may be longer than the slots)
    tok = torch.randint(0, vocab, (T,), generator=g, device=DEV, dtype=torch.int32)
    if T > 2:
        tok[1], tok[2] = -1, vocab      # no expert of theirs
    chosen, weight = torch.empty(T, top, dtype=torch.int32, device=DEV), torch.empty(T, top, device=DEV)
    ops.moe_table_route(tok, tab, top, chosen, weight)
    if not table:
        weight = torch.rand(T, top, generator=g, device=DEV) + 0.1
        if T > 4:
            chosen[4, 0] = E + 3      # out of range: skipped
    want_chosen, want_weight = chosen.clone(), weight.clone()
    if table:
        chosen.fill_(-5)
        weight.fill_(-1.0)
    act, act_s, out = torch.zeros(T * top, F, dtype=BF16, device=DEV), torch.empty(T, Fs, dtype=BF16, device=DEV), torch.empty(T, H, device=DEV)
    ops.moe_few_beside(h, w_up, down, chosen, weight, act, s_up, s_down, act_s, out, weigh_input=weigh_input,
                       **(dict(tokens=tok, table=tab) if table else {}))
    assert torch.equal(chosen, want_chosen) and torch.equal(weight, want_weight)
    x = h.double()
    _act_check(act_s, x, s_up[:Fs].double(), s_up[Fs:].double(), 1.0)
    want = act_s.double() @ s_down.double().t()
    bound = _sum_bound(act_s.double(), s_down.double())
    for r in range(T):
        for j in range(top):
            e = int(chosen[r, j])
            if not 0 <= e < E:
                continue
            f = float(weight[r, j])
            a = act[r * top + j:r * top + j + 1]
            _act_check(a, x[r:r + 1], gate[e].double(), up[e].double(), f if weigh_input else 1.0)
            one = a.double() @ down[e].double().t() * (1.0 if weigh_input else f)
            want[r] += one[0]
            bound[r] += (_sum_bound(a.double(), down[e].double()) * max(f, 1.0) + one.abs() * 2.0 ** -23)[0]
    assert ((out.double() - want).abs() <= bound + want.abs() * (top + 2) * 2.0 ** -24 + bound * 2.0 ** -20).all()


def test_which_rows():
    from kvcm_amd import ops
    w = lambda Fs, K=2048, dtype=BF16: torch.empty(2 * Fs, K, dtype=dtype, device=DEV)
    takes = lambda T, Fs, top=2, E=8, K=2048, w_=None: ops.moe_few_beside_takes(torch.empty(T, K, dtype=BF16, device=DEV), 1408, 2048, top, E, w(Fs, K) if w_ is None else w_)
    assert takes(1, 2816) and takes(8, 5632) and takes(16, 2816)
    assert not takes(9, 5632) and not takes(17, 64) and not takes(8, 2800) and not takes(16, 64, top=5) and not takes(8, 64, E=33)
    assert not takes(8, 64, w_=w(64, dtype=torch.float32))
