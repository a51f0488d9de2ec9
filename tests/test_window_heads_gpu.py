"""The window attention that takes a row's query heads together: odd sizes of heads, groups, pages and blocks against
64 bits and against the kernel it stands in for (which rows of an odd stride still take)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [dict(nh=34, nkv=2, d=8, dv=8, B=24, W=20, P=5, T=131), dict(nh=20, nkv=1, d=40, dv=56, B=8, W=64, P=1, T=200),
          dict(nh=4, nkv=4, d=128, dv=120, B=40, W=70, P=3, T=97), dict(nh=16, nkv=1, d=72, dv=128, B=48, W=0, P=0, T=700, cap=3.0, sink=True),
          dict(nh=6, nkv=2, d=64, dv=64, B=16, W=33, P=0, T=150, keep=70, slope=True), dict(nh=8, nkv=2, d=32, dv=16, B=64, W=0, P=0, T=129, chunk=50, gate=True),
          dict(nh=3, nkv=1, d=64, dv=72, B=32, W=600, P=64, T=1400, gate=True)]


def _want(q, K, V, ctx, s):
    """One row in 64 bits: q [nh, d], K / V [T, nkv, .]."""
    nh, nkv, W, P, keep, chunk = s["nh"], s["nkv"], s["W"], s["P"], s.get("keep", 0), s.get("chunk", 0)
    first = (ctx - 1) // chunk * chunk if chunk else max(0, ctx - W) if W else 0
    see = [t for t in range(ctx) if t >= first or t < keep]
    k, v, dist = K[see], V[see], torch.tensor([ctx - 1 - t for t in see], dtype=torch.float64)
    nb = (ctx - W) // P if P and W and ctx > W else 0
    if nb:
        k = torch.cat([k, K[:nb * P].reshape(nb, P, nkv, -1).mean(1)])
        v = torch.cat([v, V[:nb * P].reshape(nb, P, nkv, -1).mean(1)])
    out = []
    for h in range(nh):
        z = k[:, h // (nh // nkv)] @ q[h] * s["scale"] * s["temp"][h]
        if s.get("cap"):
            z = s["cap"] * torch.tanh(z / s["cap"])
        if s.get("slope"):
            z = z - s["slopes"][h] * dist
        m = z.max()
        p = torch.exp(z - m)
        out.append(p @ v[:, h // (nh // nkv)] / (p.sum() + (torch.exp(s["sinks"][h] - m) if s.get("sink") else 0.0)))
    return torch.stack(out)


@pytest.mark.parametrize("s", SHAPES)
def test_heads_together(s):
    from kvcm_amd import ops
    g = torch.Generator().manual_seed(s["d"] + s["T"])
    nh, nkv, d, dv, B, W, P, T = (s[k] for k in ("nh", "nkv", "d", "dv", "B", "W", "P", "T"))
    s = dict(s, scale=d ** -0.5, temp=(1 + torch.rand(nh, generator=g)), slopes=torch.rand(nh, generator=g) * 0.1, sinks=torch.randn(nh, generator=g))
    q, K, V = (torch.randn(T, n, e, generator=g).bfloat16() for n, e in ((nh, d), (nkv, d), (nkv, dv)))
    n = -(-T // B)
    order = torch.randperm(n + 3, generator=g)[:n]
    kc = torch.full((n + 3, nkv, B, d), float("nan"), dtype=torch.bfloat16)      # what no token wrote may hold anything
    vc = torch.full((n + 3, nkv, dv, B), float("nan"), dtype=torch.bfloat16)
    for t in range(T):
        kc[order[t // B], :, t % B] = K[t]
        vc[order[t // B], :, :, t % B] = V[t]
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).to(DEV)
    kc, vc, table, zeros = kc.to(DEV), vc.to(DEV), i32(order), i32([0] * T)
    pk = torch.full((n + 3, nkv, -(-B // P), d), float("nan"), device=DEV) if P else None
    pv = torch.full((n + 3, nkv, -(-B // P), dv), float("nan"), device=DEV) if P else None
    if P:
        slots = i32([int(order[t // B]) * B + t % B for t in range(T)])
        ops.pool_update(kc, vc, pk, pv, table, n, zeros, i32(range(T)), slots, nkv, d, dv, P, T)
    rows = sorted({0, 1, 7, 8, 63, 64, 65, T - 2, T - 1} | ({W - 1, W, W + max(P, 1), W + 1} if W else set()))
    rows = [r for r in rows if r < T]
    ctx = i32([r + 1 for r in rows] + [0])      # the last row has no context: its output is zero
    gate = torch.randn(len(rows) + 1, nh * dv, generator=g).to(DEV) if s.get("gate") else None

    def run(ld, at):
        k = len(at)
        buf = torch.zeros(k, ld, dtype=torch.bfloat16, device=DEV)
        buf[:, :nh * d] = torch.stack([q[rows[i]].reshape(-1) if i < len(rows) else q[0].reshape(-1) for i in at]).to(DEV)
        out = torch.full((k, nh * dv), float("nan"), dtype=torch.bfloat16, device=DEV)
        at_dev = torch.tensor(at, device=DEV)
        ops.attention_window_pool(buf, out, kc, vc, pk, pv, table, n, zeros, ctx[at_dev].contiguous(), nh, nkv, d, dv, s["scale"], W, P,
                                  head_scale=s["temp"].to(DEV), keep_first=s.get("keep", 0), softcap=s.get("cap", 0.0),
                                  dist_slope=s["slopes"].to(DEV) if s.get("slope") else None, chunk=s.get("chunk", 0),
                                  sink=s["sinks"].to(DEV) if s.get("sink") else False, gate=gate[at_dev].contiguous() if gate is not None else None)
        return out.cpu()

    every = list(range(len(rows) + 1))
    got, other = run(nh * d, every), run(nh * d + 1, every)
    assert (got[-1] == 0).all()
    want = torch.stack([_want(q[r].double(), K.double(), V.double(), r + 1, s) for r in rows]).reshape(len(rows), -1)
    if gate is not None:
        want = want * torch.sigmoid(gate[:-1].cpu().double())
    # 32-bit sums of up to T terms rounded to bfloat16 once: half a unit in the last place (2^-8) and what the sums may be off by
    sums = 2.0 ** -24 * (T + 64) * 4
    assert ((got[:-1].double() - want).abs() <= 2.0 ** -8 * want.abs() + sums).all()
    assert ((got[:-1].double() - other[:-1].double()).abs() <= 2.0 ** -7 * want.abs() + 2 * sums).all()      # one unit: each rounds for itself
    one = run(nh * d, [len(rows) - 1])      # a row alone: the same bits
    assert torch.equal(one[0], got[len(rows) - 1])
    # an infinite value that a row sees is infinite in its result
    t = rows[-1]
    vc[order[t // B], :, 0, t % B] = float("inf")
    assert torch.isinf(run(nh * d, [len(rows) - 1]).reshape(nh, dv)[:, 0]).all()


@pytest.mark.parametrize("nh,nkv", [(4, 1), (2, 2)])
def test_a_probability_of_zero_takes_nothing_of_its_value(nh, nkv):
    # one key whose score lies so far below the others' that its probability is zero in 32 bits, with a value near the largest
    from kvcm_amd import ops
    T, B, d = 40, 8, 64
    kc, vc = torch.zeros(5, nkv, B, d, dtype=torch.bfloat16), torch.ones(5, nkv, d, B, dtype=torch.bfloat16)
    kc[2, :, 3, 0], vc[2, :, :, 3] = -200.0, 1e38
    q = torch.zeros(1, nh * d, dtype=torch.bfloat16)
    q[0, ::d] = 1.0
    out = torch.zeros(1, nh * d, dtype=torch.bfloat16, device=DEV)
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).to(DEV)
    ops.attention_window_pool(q.to(DEV), out, kc.to(DEV), vc.to(DEV), None, None, i32(range(5)), 5, i32([0]), i32([T]), nh, nkv, d, d, 1.0, 0, 0)
    assert (out == 1.0).all()


@pytest.mark.parametrize("P", [1, 5, 8, 13, 16, 17, 40, 64])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_pooled_entries_of_many_rows(P, dtype):
    """Rows that all end a block, runs, and rows without a slot, in numbers whose waves look at one row or several: the mean of
    every block that ends, in ascending order, and nothing else."""
    from kvcm_amd import ops
    g = torch.Generator().manual_seed(P)
    nkv, d, dv, B, per = 2, 6, 70, 8, 3 * P
    pages = -(-per // B)
    for n, run in ((3, 1), (255, 1), (256, 1), (700, 1), (30, per)):
        kc = torch.randn(n * pages, nkv, B, d, generator=g).to(dtype).to(DEV)
        vc = torch.randn(n * pages, nkv, dv, B, generator=g).to(dtype).to(DEV)
        E = -(-B // P)
        pk, pv = torch.full((n * pages, nkv, E, d), 7.0, device=DEV), torch.full((n * pages, nkv, E, dv), 7.0, device=DEV)
        table = torch.randperm(n * pages, generator=g).to(torch.int32).reshape(n, pages)
        rows = [(s, p) for s in range(n) for p in (range(run) if run > 1 else [2 * P - 1])]
        slots = [-1 if i % 5 == 3 else int(table[s, p // B]) * B + p % B for i, (s, p) in enumerate(rows)]
        i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).to(DEV)
        ops.pool_update(kc, vc, pk, pv, table.to(DEV), pages, i32([s for s, _ in rows]), i32([p for _, p in rows]), i32(slots), nkv, d, dv, P, len(rows))
        wk, wv = torch.full_like(pk, 7.0), torch.full_like(pv, 7.0)
        k = kc[table.to(DEV).long()].permute(0, 2, 1, 3, 4).reshape(n, nkv, pages * B, d).float()      # by sequence and position
        v = vc[table.to(DEV).long()].permute(0, 2, 3, 1, 4).reshape(n, nkv, dv, pages * B).float()
        ends = [(s, p, slot // B) for (s, p), slot in zip(rows, slots) if slot >= 0 and (p + 1) % P == 0]
        for p in sorted({p for _, p, _ in ends}):
            s, page = (torch.tensor(x, device=DEV) for x in zip(*[(s, page) for s, q, page in ends if q == p]))
            entry = p // P - p // B * B // P
            ak, av = torch.zeros(len(s), nkv, d, device=DEV), torch.zeros(len(s), nkv, dv, device=DEV)
            for t in range(p - P + 1, p + 1):
                ak, av = ak + k[s, :, t], av + v[s, :, :, t]
            wk[page, :, entry], wv[page, :, entry] = ak * torch.tensor(1.0 / P, device=DEV), av * torch.tensor(1.0 / P, device=DEV)
        assert torch.equal(pk, wk) and torch.equal(pv, wv), (n, run)
