"""The chained norms' kernel of rows in registers: every count of slices around its trips, one and two branches, all groups of widths, the row's last
group partly empty, with and without what may be absent, against 64 bits.  A sum of n products in 32 bits is within n 2^-24 of the sum of their sizes; n squares under
a root, the products and the sums of each stage after it make (H / 2 + 24) 2^-24 of the terms' sizes, and an addition to the stream carries that on."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _norm(v, eps):
    return v / (v.square().mean(-1, keepdim=True) + eps).sqrt()


@pytest.mark.parametrize("H", [4, 1028, 2048, 2052, 4096, 5120, 8192])
@pytest.mark.parametrize("sa,sb", [(1, 0), (2, 0), (8, 0), (9, 0), (17, 0), (1, 1), (1, 3), (4, 2), (9, 8), (0, 0)])
def test_chain_rows(H, sa, sb):
    from kvcm_amd import ops
    g = torch.Generator(device=DEV).manual_seed(H + 100 * sa + sb)
    rand = lambda *n: torch.randn(*n, generator=g, device=DEV)
    T, eps = 5, 1e-5
    weight = lambda: torch.cat([rand(1), 1 + 0.2 * rand(H)])[1:].contiguous()
    wa, wb, wp, w = (weight() for _ in range(4))
    x0, u = rand(T, H) * 3, (H / 2 + 24) * 2.0 ** -24

    def branch(n):
        data = rand(n, T, H)
        return (data[0].contiguous() if n == 1 else ops.PartialSums(data.contiguous(), n, T, H, torch.empty(T, H, device=DEV))), data.double()

    pending, x, err = None, x0.double(), 0.0
    if sa:
        a, da = branch(sa)
        m, dm = da.sum(0), da.abs().sum(0) * sa * 2.0 ** -24
        b = None
        if sb:
            b, db = branch(sb)
            mb, dmb = db.sum(0), db.abs().sum(0) * sb * 2.0 ** -24
            ra, rb = (m.square().mean(-1, keepdim=True) + eps).sqrt(), (mb.square().mean(-1, keepdim=True) + eps).sqrt()
            na, nb = m / ra * wa.double(), mb / rb * wb.double()
            dm = 0.5 * ((dm / ra + dm.amax(-1, keepdim=True) / ra * m.abs() / ra) * wa.double().abs() + (dmb / rb + dmb.amax(-1, keepdim=True) / rb * mb.abs() / rb) * wb.double().abs()
                        + u * (na.abs() + nb.abs()))
            m = 0.5 * (na + nb)
        r = (m.square().mean(-1, keepdim=True) + eps).sqrt()
        add = m / r * wp.double()
        err = (dm / r + dm.amax(-1, keepdim=True) / r * m.abs() / r) * wp.double().abs() + u * add.abs()
        x = x + add
        err = err + x.abs() * 2.0 ** -24
        pending = ops.NormedBranches(a, wp, b, wa, wb, 0.5) if sb else ops.NormedBranches(a, wp)
    r = (x.square().mean(-1, keepdim=True) + eps).sqrt()
    want = x / r * w.double()
    top = err.amax(-1, keepdim=True) if sa else 0.0
    bound = (err / r + top / r * x.abs() / r) * w.double().abs() + u * want.abs()
    for dtype, rounding in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
        xs, out = x0.clone(), torch.empty(T, H, dtype=dtype, device=DEV)
        ops.rmsnorm_chain(xs, eps, pending=pending, weight=w, out=out)
        assert ((xs.double() - x).abs() <= err + 1e-30).all() if sa else torch.equal(xs, x0)
        assert ((out.double() - want).abs() <= bound + want.abs() * rounding + 1e-30).all()
    rows = torch.tensor([4, 0], dtype=torch.int32, device=DEV)      # gathered: the stream is left as it is
    xs, some = x0.clone(), torch.empty(2, H, dtype=torch.bfloat16, device=DEV)
    ops.rmsnorm_chain(xs, eps, pending=pending, weight=w, out=some, rows=rows)
    assert torch.equal(xs, x0) and torch.equal(some, out[rows.long()])
    plain = torch.empty(T, H, device=DEV)
    ops.rmsnorm_chain(xs, eps, pending=pending, out=plain, plain=True)
    assert torch.equal(plain, xs)
    if sa:      # the addition alone
        alone = x0.clone()
        ops.rmsnorm_chain(alone, eps, pending=pending)
        assert torch.equal(alone, xs)
