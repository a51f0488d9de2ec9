"""The routed experts' products on the matrix cores at the edges of their tiles, against 64 bits: grouped by expert (steps of many
rows) and expert by expert without grouping (a few rows)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(T, E, top, K, F, H, kind, seed, chosen=None):
    gen = torch.Generator().manual_seed(seed)
    bf = lambda *s, scale: (torch.randn(*s, generator=gen) * scale).bfloat16()
    h, up, down = bf(T, K, scale=1.0), bf(E, F, K, scale=K ** -0.5), bf(E, H, F, scale=F ** -0.5)
    gate = bf(E, F, K, scale=K ** -0.5) if kind == "silu" else None
    if chosen is None:
        chosen = torch.stack([torch.randperm(E, generator=gen)[:top] for _ in range(T)])
    return h, gate, up, down, chosen.to(torch.int32), torch.rand(T, top, generator=gen) + 0.1, torch.randn(T, H, generator=gen)


def _want(case, kind, weigh_input, add):
    """-> (the result in 64 bits, how far rounding an activation to bfloat16 may move it: half a unit of 2^-8 each, and as much
    again where the sum before it falls on the other side of a tie; with it the 32-bit sums' own error, which is smaller)."""
    h, gate, up, down, chosen, weight, base = (t.double() if t is not None and t.dtype != torch.int32 else t for t in case)
    want = base.clone() if add else torch.zeros_like(base)
    bound = torch.zeros_like(base)
    for t in range(h.shape[0]):
        for s, e in enumerate(chosen[t].tolist()):
            if not 0 <= e < up.shape[0]:
                continue
            g, x = weight[t, s], h[t]
            inner, outer = (g, 1.0) if weigh_input else (1.0, g)
            u = inner * (up[e] @ x)
            if kind == "silu":
                z = inner * (gate[e] @ x)
                a = z * torch.sigmoid(z) * u
            else:
                a = 0.5 * u * (1.0 + torch.erf(u / 2 ** 0.5)) if kind == "gelu" else torch.relu(u) ** 2
            want[t] += outer * (down[e] @ a)
            bound[t] += outer * (down[e].abs() @ a.abs()) * 2.0 ** -8
    return want, bound + 1e-5


def _run(form, case, kind, weigh_input, add, ld=None):
    from kvcm_amd import ops
    from kvcm_amd.parts.routed_parts import interleave_gate_up
    h, gate, up, down, chosen, weight, base = (t.to(DEV) if t is not None else None for t in case)
    T, K = h.shape
    E, F, _ = up.shape
    H, top = down.shape[1], chosen.shape[1]
    if kind == "silu":
        up = interleave_gate_up(gate, up)
    if ld is None:
        wide = torch.full((T, K + 24), float("nan"), dtype=torch.bfloat16, device=DEV)      # rows apart: what lies between is not read
    else:
        wide = torch.empty((T - 1) * ld + K, dtype=torch.bfloat16, device=DEV).as_strided((T, K), (ld, 1))
    wide[:, :K] = h
    act = torch.empty(T * top, F, dtype=torch.bfloat16, device=DEV)
    out = torch.full((T, H), float("nan"), device=DEV)
    how = dict(gated=kind == "silu", add=base if add else None, weigh_input=weigh_input, **({} if kind == "silu" else {"activation": kind}))
    if form == "grouped":
        order = torch.empty(T * top, dtype=torch.int32, device=DEV)
        tiles = torch.empty(ops.moe_grouped_tiles(T * top, E), dtype=torch.int32, device=DEV)
        y = torch.full((T * top, H), float("nan"), device=DEV)
        ops.moe_grouped(wide[:, :K], up, down, chosen, weight, order, tiles, act, y, out, **how)
    else:
        ops.moe_rows(wide[:, :K], up, down, chosen, weight, act, out, few=form == "few", **how)
    return out.cpu().double()


def _check(form, case, kind, weigh_input, add):
    want, bound = _want(case, kind, weigh_input, add)
    got = _run(form, case, kind, weigh_input, add)
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())
    # a row that is not finite stays alone
    bad = [case[0].clone(), *case[1:]]
    bad[0][case[0].shape[0] // 2] = float("nan")
    again = _run(form, bad, kind, weigh_input, add)
    keep = torch.arange(want.shape[0]) != want.shape[0] // 2
    assert torch.equal(again[keep], got[keep])


# one expert with 127 to 129 of the pairs (a tile's edge), K below, at and past 64 and 128, columns that end inside a tile
GROUPED = [(128, 3, 1, 64, 64, 128, "relu2", True), (129, 2, 1, 72, 48, 130, "silu", True), (127, 2, 2, 8, 40, 33, "gelu", False),
           (300, 5, 2, 136, 144, 260, "silu", False), (70, 9, 3, 200, 136, 128, "relu2", False)]


@pytest.mark.parametrize("weigh_input", [False, True])
@pytest.mark.parametrize("shape", GROUPED)
def test_grouped_tiles(shape, weigh_input):
    T, E, top, K, F, H, kind, one = shape
    chosen = torch.zeros(T, top, dtype=torch.long) if one else None
    _check("grouped", _case(T, E, top, K, F, H, kind, T + K, chosen), kind, weigh_input, not weigh_input)


# rows that lie beyond 4 GB, rows of the experts' matrices and of activations that are 8 MB apart
@pytest.mark.parametrize("shape,ld", [((40, 3, 2, 72, 48, 130, "silu"), 1 << 26), ((20, 2, 1, (1 << 22) + 8, 16, 24, "gelu"), None),
                                      ((20, 2, 1, 8, (1 << 22) + 16, 8, "relu2"), None)])
def test_grouped_rows_far_apart(shape, ld):
    T, E, top, K, F, H, kind = shape
    case = _case(T, E, top, K, F, H, kind, T + E)
    want, bound = _want(case, kind, False, True)
    got = _run("grouped", case, kind, False, True, ld)
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())


# (rows, experts, experts a row, K, F, H): one unit of 64 for eight or four waves, odd units, more than 8 and 16 pairs of one expert
# ("one"), an expert named twice by a row, and numbers that name none
FEW = [(3, 8, 2, 64, 64, 8, "silu", None), (15, 8, 2, 448, 192, 136, "relu2", None), (20, 3, 3, 128, 128, 64, "gelu", None),
       (32, 4, 2, 320, 64, 72, "silu", "one"), (9, 40, 7, 192, 128, 24, "relu2", None), (10, 6, 2, 128, 320, 16, "silu", "odd"),
       (17, 5, 1, 64, 448, 40, "gelu", "one"), (64, 8, 1, 576, 64, 8, "silu", None),
       # activations of a row, and rows, that a workgroup's LDS would not hold
       (16, 3, 2, 64, 8256, 8, "silu", None), (16, 2, 1, 16448, 64, 8, "relu2", None)]


@pytest.mark.parametrize("weigh_input", [False, True])
@pytest.mark.parametrize("shape", FEW)
def test_few_rows(shape, weigh_input):
    T, E, top, K, F, H, kind, how = shape
    chosen = None
    if how == "one":
        chosen = torch.full((T, top), E - 1)
        chosen[:, 0] = torch.arange(T) % 7 // 6 * (E - 2)      # six rows of seven choose expert 0
    elif how == "odd":
        chosen = torch.stack([torch.arange(T) % E, torch.arange(T) % 3], 1)
        chosen[2] = 4
        chosen[5, 0], chosen[7] = -1, E
    _check("few", _case(T, E, top, K, F, H, kind, T + K, chosen), kind, weigh_input, not weigh_input)


# sizes at which a row-by-row kernel, one of a few rows' two, or both run (the way whose measured time is the shorter)
@pytest.mark.parametrize("T,E,top,K,F,H,kind", [(3, 8, 2, 64, 64, 64, "silu"), (4, 16, 1, 1024, 1408, 2048, "silu"), (6, 16, 1, 1024, 1408, 2048, "silu"),
                                                (3, 2, 1, 1024, 1408, 64, "silu"), (5, 8, 2, 1024, 704, 2048, "gelu"), (15, 8, 2, 768, 512, 1024, "relu2"),
                                                (15, 8, 2, 1024, 1024, 1024, "relu2"), (11, 40, 2, 1024, 704, 2048, "silu"), (2, 8, 4, 1024, 1408, 2048, "silu"),
                                                # what a row-by-row kernel's LDS would not hold
                                                (8, 3, 2, 64, 8256, 64, "silu"), (4, 2, 1, 16448, 64, 8, "relu2")])
def test_rows_by_the_faster_kernels(T, E, top, K, F, H, kind):
    _check("rows", _case(T, E, top, K, F, H, kind, T + F), kind, False, True)


@pytest.mark.parametrize("T,K,F,H,top,E,gated,few", [
    (8, 2048, 1408, 2048, 2, 8, True, True), (16, 2048, 1408, 2048, 2, 8, True, True), (17, 2048, 1408, 2048, 2, 8, True, False),
    (16, 2048, 1408, 2048, 1, 16, True, True), (16, 2048, 1408, 2048, 1, 33, True, False), (64, 2048, 1408, 2048, 1, 16, True, False), (16, 4096, 3584, 4096, 2, 8, True, False), (15, 4096, 3584, 4096, 2, 8, True, True),
    (15, 512, 256, 512, 2, 8, True, False), (3, 2048, 1408, 2048, 1, 4, True, False), (2, 2048, 1408, 2048, 8, 8, True, False),
    (8, 2048, 1408, 2048, 2, 64, True, False), (8, 1024, 704, 2048, 2, 8, True, True), (8, 1024, 704, 2048, 2, 16, False, False), (16, 2048, 1408, 2048, 5, 32, True, False)])
def test_which_steps_a_few_rows_kernels_take(T, K, F, H, top, E, gated, few):
    from kvcm_amd import ops
    assert bool(ops.lib().kvcm_moe_few_takes(T, K, F, H, top, E, int(gated))) == few


@pytest.mark.parametrize("T,top,H,F", [(16, 2, 64, 8256), (32, 2, 64, 8256), (20, 1, 16448, 64)])
def test_layers_wider_than_a_workgroups_local_memory(T, top, H, F):
    """the layer takes rows and activations of any width from 16 rows on, by whichever kernels"""
    from kvcm_amd import ops
    from kvcm_amd.parts.base import BuildContext
    from kvcm_amd.parts.routed_parts import RoutedExperts
    E = 3
    h, _, up, down, chosen, _, _ = case = _case(T, E, top, H, F, H, "relu2", T + F)
    part = RoutedExperts({"experts": E, "top": top, "ff": F, "routing": "table", "vocab_size": T}, "",
                         BuildContext(torch.bfloat16, torch.device(DEV), H, 16, ops))
    part.bind({"table": chosen.to(DEV), "w_up": up.view(E * F, H).to(DEV), "w_down": down.view(E * H, F).to(DEV)})

    class Step:
        rows, limits, tune_products, tokens = T, None, None, torch.arange(T, dtype=torch.int32, device=DEV)

        def ws(self, name, shape, dtype=torch.bfloat16):
            return torch.empty(shape, dtype=dtype, device=DEV)

        def flat(self, name, numel, dtype=torch.float32):
            return torch.empty(numel, dtype=dtype, device=DEV)

    got = part.forward(Step(), h.to(DEV)).cpu().double()
    want, bound = _want((*case[:5], torch.full((T, top), 1.0 / top), case[6]), "relu2", False, False)
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())
