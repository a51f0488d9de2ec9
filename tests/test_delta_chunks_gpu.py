"""The delta rule in matrix form (csrc/hip/delta_chunks.hip) against the plain recurrence: chunks of 64 and 32 rows that end anywhere, runs that
begin in the middle of a sequence, heads that end inside a tile, rows that begin at any float, dead slots, scratch for a part of a run."""
import numpy as np
import pytest
import torch

import plain_kasuvik as plain
from test_kasuvik_gpu import Step, dev

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("turns", [False, True])
@pytest.mark.parametrize("d,dv,shift", [(64, 64, 0), (64, 50, 1), (33, 64, 1), (60, 20, 0), (128, 128, 0), (100, 17, 1), (65, 128, 0)])
def test_long_runs_against_the_plain_recurrence(d, dv, shift, turns, monkeypatch):
    from kvcm_amd import ops
    monkeypatch.setattr(ops, "delta_in_chunks", lambda *a: True)
    rng = np.random.default_rng(d + dv)
    heads, parts = 2, ((256, 1, 129, 64), (63, 321, 128, 7), (257, 192, 1, 385))
    seqs, D = len(parts[0]), 2 * d
    lowest = np.exp(-np.exp(-0.5))
    data = []
    for n in (sum(x[i] for x in parts) for i in range(seqs)):
        q = {"r": rng.normal(size=(n, heads, d)), "k": rng.normal(size=(n, heads, d)), "v": rng.normal(size=(n, heads, dv)),
             "w": np.where(rng.random((n, heads, d)) < 0.3, lowest, rng.uniform(lowest, 1.0, size=(n, heads, d))), "a": rng.uniform(0, 1, size=(n, heads, d))}
        q["w"][:, 1, ::2] = lowest ** rng.uniform(0, 0.02, size=(n, heads, d))[:, 1, ::2]      # (channels that keep for long beside some that forget at once)
        q["u"] = q["k"] / np.sqrt((q["k"] ** 2).sum(-1, keepdims=True) + 1e-6)
        data.append(q)
    want = [plain.delta_rule(q["r"], q["k"], q["v"], q["w"], q["a"]) for q in data]
    S, at = torch.full((seqs, heads, d, dv), 9.0, device=DEV), [0] * seqs
    for part in parts:
        st = Step([(i, at[i], n) for i, n in enumerate(part)] + [(0, 5, 140)])
        st.max_run = max(part)
        st.state_slots[-1] = -1      # a padding sequence beside them
        cat = lambda f, c: dev(np.concatenate([f(q)[at[i]:at[i] + n].reshape(n, -1) for i, (q, n) in enumerate(zip(data, part))] + [rng.uniform(0.6, 1, (140, c))]))
        r, k, v = (cat(lambda q, x=x: q[x], c) for x, c in (("r", D), ("k", D), ("v", heads * dv)))
        packed = torch.full((st.rows, 2 * D + heads * dv + 2 + shift), float("nan"), device=DEV)[:, shift:]
        packed[:, :D], packed[:, D:2 * D], packed[:, 2 * D:2 * D + heads * dv] = r, k, v
        w, au, u = cat(lambda q: q["w"], D), cat(lambda q: q["a"] * q["u"], D), cat(lambda q: q["u"], D)
        one = int(ops.lib().kvcm_delta_carry_floats(st.seqs, 1, heads, d))
        carry = torch.full((3 * one if turns else ops.delta_carry_floats(st.rows, st.seqs, heads, d),), float("nan"), device=DEV)
        o = torch.full((st.rows, heads * dv + shift), float("nan"), device=DEV)
        ops.delta_scan(packed, packed[:, D:], packed[:, 2 * D:], w, au, u, o, S, st, heads, d, dv, carry=carry)
        row, got = 0, o[:, :heads * dv].double().cpu().numpy()
        for i, n in enumerate(part):
            ref = want[i][at[i]:at[i] + n].reshape(n, -1)
            # as the walk's: sums of up to 128 keys a row, handed on by a state that forgets
            np.testing.assert_allclose(got[row:row + n], ref, atol=5e-5 * max(1.0, np.abs(ref).max()), err_msg=f"sequence {i} from {at[i]}")
            row, at[i] = row + n, at[i] + n
        assert not got[row:].any()


@pytest.mark.gpu
def test_the_line_between_the_forms():
    from kvcm_amd import ops
    def step(*runs):
        st = Step([(i, 0, n) for i, n in enumerate(runs)])
        st.max_run = max(runs)
        return st
    assert ops.delta_in_chunks(step(192), 4, 64, 64) and not ops.delta_in_chunks(step(191), 4, 64, 64)
    assert ops.delta_in_chunks(step(128), 4, 65, 128) and not ops.delta_in_chunks(step(127), 4, 65, 128)
    assert ops.delta_in_chunks(step(192, 192, 192), 32, 64, 64) and not ops.delta_in_chunks(step(192, 192, 192), 33, 64, 64)
    for heads, d, dv, takes in ((4, 128, 128, True), (4, 129, 64, False), (4, 32, 32, False), (4, 33, 64, True), (4, 64, 65, False), (1 << 17, 128, 64, False)):
        assert ops.delta_in_chunks(step(200), heads, d, dv) == takes
    assert not ops.delta_in_chunks(step(200), 4, 64, 64, True)
    assert ops.delta_in_chunks(step(200, 1), 4, 64, 64) and not ops.delta_in_chunks(step(200, 1, 1), 4, 64, 64)      # (runs of similar lengths)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 100])
@pytest.mark.parametrize("mean", [0, 1, 2, 5])
def test_keys_that_resemble_each_other(d, mean):
    """Keys and values around a common row, removed at nearly the whole rate: what a chunk learns is small beside what it says, and the form's errors
    against 64 bits are no larger than the walk's."""
    from kvcm_amd import ops
    heads, T = 8, 512
    rng = np.random.default_rng(100 * d + mean)
    f32 = lambda x: x.astype(np.float32)
    k, v = (f32(rng.normal(size=(T, heads, d)) + mean * rng.normal(size=(1, heads, d))) for _ in range(2))
    r, u = f32(rng.normal(size=(T, heads, d))), f32(k / np.sqrt((k.astype(np.float64) ** 2).sum(-1, keepdims=True)))
    sigmoid = lambda x: 1 / (1 + np.exp(-x))
    w = f32(np.exp(-np.exp(-0.5) * sigmoid(rng.normal(size=(T, heads, d)) - 2)))
    au = f32(sigmoid(rng.normal(size=(T, heads, d)) + 4) * u)
    r8, k8, v8, w8, a8, u8 = (x.astype(np.float64) for x in (r, k, v, w, au, u))
    want, state = np.zeros((T, heads, d)), np.zeros((heads, d, d))
    for i in range(T):
        z = np.einsum("hk,hkv->hv", u8[i], state)
        state = w8[i][:, :, None] * state - a8[i][:, :, None] * z[:, None] + k8[i][:, :, None] * v8[i][:, None]
        want[i] = np.einsum("hk,hkv->hv", r8[i], state)
    st = Step([(0, 0, T)])
    st.max_run = T
    ops_in = [dev(x.reshape(T, heads * d)) for x in (r, k, v, w, au, u)]
    errors = []
    for carry in (None, torch.empty(ops.delta_carry_floats(T, 1, heads, d), device=DEV)):
        o, S = torch.empty(T, heads * d, device=DEV), torch.zeros(1, heads, d, d, device=DEV)
        ops.delta_scan(*ops_in, o, S, st, heads, d, d, carry=carry)
        rel = lambda x, y: np.linalg.norm(x.double().cpu().numpy().reshape(-1) - y.reshape(-1)) / np.linalg.norm(y)
        errors.append((rel(o, want), rel(S, state)))
    # root mean squares of T x heads x d and of heads x d x d roundings: alike to a few parts in a hundred from one draw to another
    for walk, chunks in zip(*errors):
        assert chunks <= 1.05 * walk, errors


@pytest.mark.gpu
@pytest.mark.parametrize("heads,d,dv,runs", [(32, 64, 64, (1100, 700)), (32, 64, 33, (1024, 1)), (40, 48, 48, (509, 100, 509)), (16, 128, 128, (600, 333, 32)),
                                             (24, 90, 128, (777, 1))])
def test_chunks_one_after_the_other(heads, d, dv, runs):
    """More chunks than workgroups at once: outputs and states of steps that take all of the scratch, each run in places of its own, against 64 bits, and
    bit for bit those of scratch for some chunks of every sequence, which a workgroup's turns do not divide."""
    from kvcm_amd import ops
    T, D = sum(runs), heads * d
    g = torch.Generator(device=DEV).manual_seed(heads + d)
    r, k, v = (torch.randn(T, heads, c, generator=g, device=DEV) for c in (d, d, dv))
    u = k / (k.norm(dim=-1, keepdim=True) + 1e-6)
    w = torch.exp(-0.6065306 * torch.rand(T, heads, d, generator=g, device=DEV) ** 3)
    au = torch.rand(T, heads, d, generator=g, device=DEV) * u
    first = torch.randn(len(runs), heads, d, dv, generator=g, device=DEV)
    r8, k8, v8, w8, a8, u8 = (x.double() for x in (r, k, v, w, au, u))
    state, want, row = first.double(), torch.empty(T, heads, dv, dtype=torch.float64, device=DEV), 0
    for s, n in enumerate(runs):
        for i in range(row, row + n):
            z = (u8[i].unsqueeze(-1) * state[s]).sum(1, keepdim=True)
            state[s] = w8[i].unsqueeze(-1) * state[s] - a8[i].unsqueeze(-1) * z + k8[i].unsqueeze(-1) * v8[i].unsqueeze(1)
            want[i] = (r8[i].unsqueeze(-1) * state[s]).sum(1)
        row += n
    st = Step([(i, 5, n) for i, n in enumerate(runs)])
    st.max_run = max(runs)
    assert ops.delta_in_chunks(st, heads, d, dv) or 2 * T < len(runs) * max(runs)
    full, one = ops.delta_carry_floats(T, len(runs), heads, d), int(ops.lib().kvcm_delta_carry_floats(len(runs), 1, heads, d))
    flat, got = (lambda x: x.reshape(T, -1).contiguous()), []
    for floats in (full, 5 * one, 3 * one):
        o, S = torch.full((T, heads * dv), float("nan"), device=DEV), first.clone()
        carry = torch.full((floats,), float("nan"), device=DEV)
        a = [flat(x) for x in (r, k, v, w, au, u)]
        ops._call("kvcm_delta_chunks", ops._ptr(a[0]), D, ops._ptr(a[1]), D, ops._ptr(a[2]), heads * dv, ops._ptr(a[3]), ops._ptr(a[4]), ops._ptr(a[5]),
                  ops._ptr(o), heads * dv, ops._ptr(S), ops._ptr(st.run_start), ops._ptr(st.seq_start), ops._ptr(st.state_slots), len(runs), heads, d, dv, T,
                  max(runs), ops._ptr(carry), floats, ops._stream())
        got.append((o, S))
        assert torch.equal(o, got[0][0]) and torch.equal(S, got[0][1])
    # as the walk's: sums of up to 128 keys a row, handed on by a state that forgets
    for x, y in zip(got[0], (want, state)):
        assert float((x.double().view_as(y) - y).abs().max()) < 5e-5 * max(1.0, float(y.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["v", "k", "r", "au", "u"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("d", [64, 100])
def test_what_is_not_finite_stays_behind_its_row(d, value, what):
    """Rows in front of a value that is not finite are as if it were not there, whatever the place of its row in a chunk; from it on, what the walk says is finite is."""
    from kvcm_amd import ops
    heads, runs = 2, (200, 192, 256)
    T, D = sum(runs), heads * d
    st = Step([(i, 5, n) for i, n in enumerate(runs)])
    st.max_run = max(runs)
    g = torch.Generator(device=DEV).manual_seed(d)
    a = {x: torch.randn(T, D, generator=g, device=DEV) for x in ("r", "k", "v")}
    a["w"] = torch.exp(-0.6065306 * torch.rand(T, D, generator=g, device=DEV))
    a["u"] = a["k"] / d ** 0.5
    a["au"] = a["u"] * torch.rand(T, D, generator=g, device=DEV)
    first = torch.randn(len(runs), heads, d, d, generator=g, device=DEV)
    clean = {x: y.clone() for x, y in a.items()}
    for row, channel in ((75, 3), (200 + 64 + 30, d + 1), (392 + 37, 20)):      # (in the second head's first run of rows too)
        a[what][row, channel] = value
    out = []
    for q, carry in ((clean, True), (a, True), (a, False)):
        o, S = torch.full((T, D), 7.0, device=DEV), first.clone()
        kw = dict(carry=torch.full((ops.delta_carry_floats(T, len(runs), heads, d),), float("nan"), device=DEV)) if carry else {}
        ops.delta_scan(q["r"], q["k"], q["v"], q["w"], q["au"], q["u"], o, S, st, heads, d, d, **kw)
        out.append((o, S))
    (same, state), (o, S), (walk, walked) = out
    assert torch.isfinite(same).all() and not torch.isfinite(o).all()
    # where the walk's numbers are finite, ours are, and as near as two orders of the same sums are (as above)
    for x, y, ref in ((o, walk, same), (S, walked, state)):
        assert torch.equal(torch.isfinite(x), torch.isfinite(y))
        ok = torch.isfinite(y)
        assert float((x[ok] - y[ok]).abs().max()) < 1e-4 * float(ref.abs().max())
