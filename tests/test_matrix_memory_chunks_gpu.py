"""The matrix memory in matrix form (csrc/hip/mlstm_chunks.hip) against the plain recurrence: chunks of 64 rows and pieces of 128 that end
anywhere, runs that begin in the middle of a sequence, keys and values that end inside a tile, rows that begin at any float, dead slots."""
import numpy as np
import pytest
import torch

import plain_furapel as plain
from test_kasuvik_gpu import Step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("d,dv,shift", [(64, 64, 0), (64, 130, 0), (16, 6, 1), (100, 20, 0), (128, 72, 0), (20, 33, 1), (65, 4, 0)])
def test_long_runs_against_the_plain_recurrence(d, dv, shift):
    from kvcm_amd import ops
    rng = np.random.default_rng(d + dv)
    heads, cap, parts = 2, 12.0, ((256, 1, 129, 64), (63, 321, 128, 7), (257, 192, 1, 385))
    seqs = len(parts[0])
    total = [sum(x[i] for x in parts) for i in range(seqs)]
    # positive keys and queries: the divisor n . q has no cancellation; then sums of up to 256 products and 64 rows in up to three pieces stay
    # within 3e-5 of 32-bit rounding (twice 256 steps of 2^-24)
    data = [[np.abs(rng.normal(size=(n, heads, d))), np.abs(rng.normal(size=(n, heads, d))), rng.normal(size=(n, heads, dv)),
             rng.normal(size=(n, heads)) * 4, rng.normal(size=(n, heads)) * 4 + 2] for n in total]
    bi, bf = rng.normal(size=heads), rng.normal(size=heads)
    want = []
    for q, k, v, gi, gf in data:
        o = np.zeros((q.shape[0], heads, dv))
        for a in range(heads):
            o[:, a], _ = plain.matrix_memory(q[:, a] * d ** -0.5, k[:, a], v[:, a], plain.soft_cap(gi[:, a] + bi[a], cap),
                                             plain.log_sigmoid(plain.soft_cap(gf[:, a] + bf[a], cap)))
        want.append(o.reshape(-1, heads * dv))

    def dev(x):
        return torch.tensor(np.asarray(x), dtype=torch.float32, device=DEV)

    # (a dead slot beside them: its rows are zero, and it has no state)
    S = torch.full((seqs, heads, d, dv), 9.0, device=DEV)
    N, M = torch.full((seqs, heads, d), -3.0, device=DEV), torch.full((seqs, heads), 50.0, device=DEV)
    cols = np.cumsum([0, heads * d, heads * d, heads * dv, heads])
    at = [0] * seqs
    for part in parts:
        st = Step([(i, at[i], n) for i, n in enumerate(part)] + [(0, 5, 140)])
        st.max_run = max(part)
        slots = st.state_slots.clone()
        slots[-1] = -1
        st.state_slots = slots
        rows = np.concatenate([np.concatenate([x[at[i]:at[i] + n].reshape(n, -1) for x in data[i]], 1) for i, n in enumerate(part)]
                              + [rng.normal(size=(140, cols[-1] + heads))], 0)
        packed = torch.full((rows.shape[0], rows.shape[1] + 2 + shift), float("nan"), device=DEV)[:, shift:]
        packed[:, :rows.shape[1]] = dev(rows)
        x = [packed[:, lo:] for lo in cols]
        assert ops.mlstm_in_chunks(st, d) and not ops.mlstm_in_chunks(st, d, True)
        carry = torch.full((ops.mlstm_carry_floats(st.rows, st.seqs, heads, d, dv),), float("nan"), device=DEV)
        coef, o = torch.empty(st.rows, 4 * heads, device=DEV), torch.full((st.rows, heads * dv), float("nan"), device=DEV)
        ops.mlstm_scan(*x, dev(bi), dev(bf), cap, d ** -0.5, coef, torch.empty(st.seqs * heads * d, device=DEV), o, S, N, M, st, heads, d, dv,
                       carry=carry)
        row = 0
        for i, n in enumerate(part):
            ref = want[i][at[i]:at[i] + n]
            np.testing.assert_allclose(o[row:row + n].cpu().numpy(), ref, atol=3e-5 * max(1.0, np.abs(ref).max()), err_msg=f"sequence {i} from {at[i]}")
            row, at[i] = row + n, at[i] + n
        assert not bool(o[row:].any())


def test_the_line_between_the_forms():
    from kvcm_amd import ops
    short, long = Step([(0, 0, 255), (1, 0, 3)]), Step([(0, 0, 256), (1, 0, 3)])
    short.max_run, long.max_run = 255, 256
    assert not ops.mlstm_in_chunks(short, 64) and ops.mlstm_in_chunks(long, 128) and not ops.mlstm_in_chunks(long, 129)


@pytest.mark.parametrize("what", ["q", "k", "v"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("d,dv", [(64, 64), (100, 20)])
def test_what_is_not_finite_stays_behind_its_row(d, dv, value, what):
    """Rows in front of a value that is not finite are as if it were not there, whatever the place of its row in a chunk; from it on, what the walk says is finite is."""
    from kvcm_amd import ops
    heads, runs = 2, (300, 200, 256)
    T = sum(runs)
    st = Step([(i, 5, n) for i, n in enumerate(runs)])
    st.max_run = max(runs)
    g = torch.Generator(device=DEV).manual_seed(d)
    a = {x: torch.randn(T, heads * c, generator=g, device=DEV).abs() for x, c in (("q", d), ("k", d), ("v", dv))}      # (a divisor without cancellation)
    gates = torch.randn(2, T, heads, generator=g, device=DEV)
    first = [torch.rand(len(runs), heads, *c, generator=g, device=DEV) for c in ((d, dv), (d,), ())]
    clean = {x: y.clone() for x, y in a.items()}
    for row, channel in ((75, 3), (300 + 64 + 30, heads * (dv if what == "v" else d) - 2), (500 + 37, 9)):
        a[what][row, channel] = value
    out = []
    for q, carry in ((clean, True), (a, True), (a, False)):
        o, states = torch.full((T, heads * dv), 7.0, device=DEV), [x.clone() for x in first]
        kw = dict(carry=torch.full((ops.mlstm_carry_floats(T, len(runs), heads, d, dv),), float("nan"), device=DEV)) if carry else {}
        ops.mlstm_scan(q["q"], q["k"], q["v"], gates[0], gates[1], torch.zeros(heads, device=DEV), torch.full((heads,), 4.0, device=DEV), 15.0, d ** -0.5,
                       torch.empty(T, 4 * heads, device=DEV), torch.empty(len(runs) * heads * d, device=DEV), o, *states, st, heads, d, dv, **kw)
        out.append((o, *states))
    assert all(torch.isfinite(x).all() for x in out[0]) and not torch.isfinite(out[1][0]).all()
    for ref, x, y in zip(*out):
        assert torch.equal(torch.isfinite(x), torch.isfinite(y))
        ok = torch.isfinite(y)
        assert float((x[ok] - y[ok]).abs().max()) < 6e-5 * float(ref.abs().max())      # both within 3e-5 of the recurrence, as above


@pytest.mark.parametrize("d", [64, 128])
def test_errors_of_long_runs_are_the_walks(d):
    """Runs of many pieces that are gone on with: outputs, states, normalizers and maxima against 64 bits, with errors as the walk's."""
    from kvcm_amd import ops
    heads, parts, cap = 16, ((513, 1025, 1500), (300, 257, 700)), 15.0
    seqs, total = 3, [813, 1282, 2200]
    g = torch.Generator(device=DEV).manual_seed(d)
    draw = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    data = [[draw(n, heads, d) + draw(1, heads, d), draw(n, heads, d) + draw(1, heads, d), draw(n, heads, d), draw(n, heads), draw(n, heads)] for n in total]
    bi, bf = draw(heads) * 0.1 - 1, torch.linspace(3, 6, heads, device=DEV)
    want, states = [], []
    for q, k, v, gi, gf in data:
        soft = lambda x: cap * torch.tanh(x.double() / cap)
        li, lf = soft(gi + bi), torch.nn.functional.logsigmoid(soft(gf + bf))
        S, n, m = (torch.zeros(heads, *x, dtype=torch.float64, device=DEV) for x in ((d, d), (d,), ()))
        o = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        q, k, v = q.double() * d ** -0.5, k.double(), v.double()
        for t in range(q.shape[0]):
            m1 = torch.maximum(lf[t] + m, li[t])
            keep, take, m = torch.exp(lf[t] + m - m1), torch.exp(li[t] - m1), m1
            S = keep[:, None, None] * S + (take[:, None] * k[t]).unsqueeze(2) * v[t].unsqueeze(1)
            n = keep[:, None] * n + take[:, None] * k[t]
            o[t] = (q[t].unsqueeze(2) * S).sum(1) / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        want.append(o)
        states.append((S, n, m))
    errors = []
    for chunks in (False, True):
        S, N, M = (torch.full((seqs, heads, *x), 7.0, device=DEV) for x in ((d, d), (d,), ()))
        at, outs = [0] * seqs, [[] for _ in range(seqs)]
        for part in parts:
            st = Step([(i, at[i], n) for i, n in enumerate(part)])
            st.max_run = max(part)
            rows = [torch.cat([x[j][at[i]:at[i] + n].flatten(1) for i, (x, n) in enumerate(zip(data, part))]) for j in range(5)]
            o = torch.full((st.rows, heads * d), float("nan"), device=DEV)
            kw = dict(carry=torch.full((ops.mlstm_carry_floats(st.rows, seqs, heads, d, d),), float("nan"), device=DEV)) if chunks else {}
            assert ops.mlstm_in_chunks(st, d)
            ops.mlstm_scan(*rows, bi, bf, cap, d ** -0.5, torch.empty(st.rows, 4 * heads, device=DEV), torch.empty(seqs * heads * d, device=DEV), o, S, N, M, st,
                           heads, d, d, **kw)
            for i, x in enumerate(o.split(list(part))):
                outs[i].append(x.view(-1, heads, d))
                at[i] += part[i]
        rel = lambda x, y: float((x.double() - y).norm() / y.norm())
        errors.append((rel(torch.cat([torch.cat(x) for x in outs]), torch.cat(want)), *(rel(x, torch.stack([y[j] for y in states])) for j, x in enumerate((S, N, M)))))
    walk, chunks = errors
    assert walk[0] < 3e-5 and max(walk[1:]) < 3e-6, errors      # (the outputs' divisor n . q cancels)
    # a state's error is that of the factors, which the forms share; what each adds is a few parts in a hundred of it
    assert all(x <= 1.03 * y for x, y in zip(chunks, walk)), errors


def test_the_line_where_the_walk_is_the_faster():
    """Single tokens beside a run, heads of few keys, many runs: the form whose measured time is the smaller (us, walk / matrix form)."""
    from kvcm_amd import ops

    def takes(heads, dk, dv, runs):
        st = Step([(i, 5, n) for i, n in enumerate(runs)])
        st.max_run = max(runs)
        return ops.mlstm_in_chunks(st, dk, False, heads, dv)

    one = [1]
    for heads, dk, dv, runs, so in ((32, 64, 64, [256], True),                    # 54 / 49
                                    (32, 64, 64, [256] + 7 * one, True),          # 90 / 63
                                    (32, 64, 64, [256] + 31 * one, False),        # 94 / 103
                                    (32, 64, 64, [256] + 63 * one, False),        # 100 / 167
                                    (32, 64, 64, [1024] + 31 * one, True),        # 311 / 125
                                    (32, 64, 64, [256] * 32, True),               # 335 / 284
                                    (32, 128, 128, [256], True),                  # 90 / 66
                                    (32, 128, 128, [256] + 7 * one, False),       # 96 / 110
                                    (32, 128, 128, [1024] + 31 * one, False),     # 318 / 358
                                    (32, 128, 64, [256] + 7 * one, False),        # 73 / 80
                                    (32, 128, 128, [256] * 4, True),              # 203 / 124
                                    (64, 16, 16, [256], True),                    # 54 / 44
                                    (64, 16, 16, [256] * 4, False),               # 57 / 66
                                    (64, 16, 16, [256] * 32, False),              # 107 / 341
                                    (64, 16, 16, [1024] + 31 * one, True),        # 172 / 135
                                    (8, 64, 64, [256] + 63 * one, True),          # 89 / 77
                                    (32, 32, 32, [256] * 16, False)):             # 88 / 114
        assert takes(heads, dk, dv, runs) == so, (heads, dk, dv, len(runs), max(runs))


def test_scratch_is_bounded_and_longer_pieces_do():
    from kvcm_amd import ops
    size = lambda rows, seqs, heads, d, piece: int(ops.lib().kvcm_mlstm_carry_floats(rows, seqs, heads, d, d, piece))
    for rows, seqs, heads, d in ((2048, 1, 32, 64), (65536, 1, 32, 128), (65536, 256, 32, 128), (1 << 20, 4, 32, 64), (8192, 64, 64, 128)):
        floats = ops.mlstm_carry_floats(rows, seqs, heads, d, d)
        assert floats <= max(ops.MLSTM_CARRY, 2 * (seqs + 1) * heads * (d * d + d + 1))
        assert ops.mlstm_piece(rows, seqs, heads, d, d, floats) >= ops.MLSTM_PIECE and size(rows, seqs, heads, d, ops.mlstm_piece(rows, seqs, heads, d, d, floats)) <= floats
        assert floats == size(rows, seqs, heads, d, ops.MLSTM_PIECE) or floats < size(rows, seqs, heads, d, ops.MLSTM_PIECE)
    heads, d, runs = 3, 64, (1100, 300, 513)
    T = sum(runs)
    st = Step([(i, 5, n) for i, n in enumerate(runs)])
    st.max_run = max(runs)
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.rand(T, heads * d, generator=g, device=DEV) for _ in range(3))      # (a divisor without cancellation)
    gates, first, out = torch.randn(2, T, heads, generator=g, device=DEV), [torch.rand(3, heads, *c, generator=g, device=DEV) for c in ((d, d), (d,), ())], []
    for piece in (128, 256, 512, 2048):
        floats, o, states = size(T, 3, heads, d, piece), torch.full((T, heads * d), float("nan"), device=DEV), [x.clone() for x in first]
        assert ops.mlstm_piece(T, 3, heads, d, d, floats) == piece
        ops.mlstm_scan(q, k, v, gates[0], gates[1], torch.zeros(heads, device=DEV), torch.full((heads,), 4.0, device=DEV), 15.0, d ** -0.5,
                       torch.empty(T, 4 * heads, device=DEV), torch.empty(3 * heads * d, device=DEV), o, *states, st, heads, d, d,
                       carry=torch.full((floats,), float("nan"), device=DEV))
        out.append((o, *states))
    for got in out[1:]:
        for x, y in zip(got, out[0]):
            assert float((x - y).abs().max()) < 6e-5 * float(y.abs().max())      # both within 3e-5 of the recurrence, as above
    with pytest.raises(RuntimeError):
        ops.mlstm_scan(q, k, v, gates[0], gates[1], torch.zeros(heads, device=DEV), torch.full((heads,), 4.0, device=DEV), 15.0, d ** -0.5,
                       torch.empty(T, 4 * heads, device=DEV), torch.empty(3 * heads * d, device=DEV), o, *states, st, heads, d, d,
                       carry=torch.empty(3 * heads * d * d, device=DEV))
