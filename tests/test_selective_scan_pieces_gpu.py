"""The selective scan in pieces of 32, 64 and 128 rows (csrc/hip/selective_scan.hip, bfloat16): runs and portions that end at a piece's
edges, both ways to deal the channels out, against the plain recurrence; and the rules that choose."""
import numpy as np
import pytest
import torch

import plain_kasuvik as plain
from test_kasuvik_gpu import Step, dev

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("piece", [32, 64, 128])
@pytest.mark.parametrize("C,N", [(257, 16), (1290, 16), (1300, 8)])
def test_pieces_against_the_plain_recurrence(C, N, piece, monkeypatch):
    from kvcm_amd import ops
    monkeypatch.setattr(ops, "scan_piece", lambda *a: piece)
    rng = np.random.default_rng(C + piece)
    parts = ((129, 31, 1, 64, 192), (65, 33, 128, 191, 4))
    grid = lambda a: torch.tensor(a).to(torch.bfloat16).double().numpy()
    data = [(grid(rng.normal(size=(n, C))), rng.normal(size=(n, C)), rng.normal(size=(n, C)) - 1.0, rng.normal(size=(n, 2 * N)))
            for n in map(sum, zip(*parts))]
    a_log, dsk, db = np.log(rng.uniform(0.3, 4.0, size=(C, N))), rng.normal(size=C), rng.normal(size=C)
    want = [plain.selective_scan(x, plain.softplus(dtl + db), -np.exp(a_log), bc[:, :N], bc[:, N:], dsk) * plain.silu(z)
            for x, z, dtl, bc in data]
    state, at = torch.full((len(data), C, N), 5.0, device=DEV), [0] * len(data)
    for part in parts:
        step = Step([(i, at[i], n) for i, n in enumerate(part)] + [(0, 7, 40)])
        step.max_run = max(part)
        step.state_slots[-1] = -1      # a padding sequence beside them
        pad = np.full((40, C), np.nan)
        cat = lambda j, pad=pad: dev(np.concatenate([x[j][at[i]:at[i] + n] for i, (x, n) in enumerate(zip(data, part))] + [pad]))
        out = torch.full((step.rows, C), float("nan"), dtype=torch.bfloat16, device=DEV)
        carry = torch.full(((step.rows // piece + step.seqs + 1) * C * (N + 1) + ops.selective_scan_carry_floats(step.rows, step.seqs, C, N),),
                           float("nan"), device=DEV)
        ops.selective_scan(cat(0).to(torch.bfloat16), cat(2), dev(db), cat(3, pad[:, :2 * N]), 0, N, dev(a_log), dev(dsk), cat(1), out, state,
                           step, prepare=True, carry=carry)
        row = 0
        for i, n in enumerate(part):      # (half a unit of 8 bits of the largest)
            ref = want[i][at[i]:at[i] + n]
            np.testing.assert_allclose(out[row:row + n].double().cpu().numpy(), ref, atol=2.0 ** -8 * max(1.0, np.abs(ref).max()))
            row, at[i] = row + n, at[i] + n
        assert not bool(out[row:].any())


@pytest.mark.gpu
def test_step_sizes_and_gates_that_are_made_already(monkeypatch):
    """The entry point with prepared rows and pieces: what it makes itself, within the result's own rounding."""
    from kvcm_amd import ops
    g = torch.Generator().manual_seed(3)
    T, C, N = 300, 1800, 16
    x, z, dt = (torch.randn(T, C, generator=g).to(DEV) for _ in range(3))
    bc, a_log, dsk, db = (torch.randn(*n, generator=g).to(DEV) for n in ((T, 2 * N), (C, N), (C,), (C,)))
    step, call = Step([(0, 0, T)]), ops._call
    step.max_run = T
    got = []
    for made in (False, True):
        def entry(name, *args, made=made):
            args = list(args)
            if name == "kvcm_selective_scan":
                if made:
                    call("kvcm_scan_prepare", *args[3:6], *args[12:14], T, C, args[-1])
                args[23] = int(made)
            return call(name, *args)
        monkeypatch.setattr(ops, "_call", entry)
        out, state = torch.empty(T, C, dtype=torch.bfloat16, device=DEV), torch.zeros(1, C, N, device=DEV)
        carry = torch.empty(ops.selective_scan_carry_floats(T, 1, C, N), device=DEV)
        ops.selective_scan(x.bfloat16(), dt.clone(), db, bc, 0, N, a_log, dsk, z.clone(), out, state, step, prepare=True, carry=carry)
        got.append((out.float(), state))
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=0, atol=2.0 ** -8 * float(b.abs().max()))


@pytest.mark.gpu
def test_scratch_for_the_longest_pieces_is_enough():
    """Scratch sized for pieces of SCAN_PIECE rows is taken where shorter ones would be the choice; less is refused."""
    from kvcm_amd import ops
    g = torch.Generator().manual_seed(4)
    T, C, N = 700, 900, 16
    x, z, dt = (torch.randn(T, C, generator=g).to(DEV) for _ in range(3))
    bc, a_log, dsk, db = (torch.randn(*n, generator=g).to(DEV) for n in ((T, 2 * N), (C, N), (C,), (C,)))
    step, got = Step([(0, 0, T)]), []
    step.max_run = T
    assert ops.scan_piece(T, C, torch.bfloat16) < ops.SCAN_PIECE
    least = ops.selective_scan_carry_floats(T, 1, C, N, ops.SCAN_PIECE)
    for floats in (ops.selective_scan_carry_floats(T, 1, C, N), least, least - 1):
        out, state = torch.empty(T, C, dtype=torch.bfloat16, device=DEV), torch.zeros(1, C, N, device=DEV)
        call = lambda: ops.selective_scan(x.bfloat16(), dt.clone(), db, bc, 0, N, a_log, dsk, z.clone(), out, state, step, prepare=True,
                                          carry=torch.full((floats,), float("nan"), device=DEV))
        if floats < least:
            with pytest.raises(Exception, match="too small"):
                call()
        else:
            call()
            got.append((out.float(), state))
    for a, b in zip(*got):      # (half a unit of 8 bits of the largest, each)
        torch.testing.assert_close(a, b, rtol=0, atol=2.0 ** -8 * float(b.abs().max()))


def test_the_scratch_holds_the_pieces_of_every_smaller_step():
    from kvcm_amd import ops
    for C, N, seqs, most in ((4096, 16, 3, 32768), (8192, 16, 1, 5000), (64, 8, 9, 40000), (1, 8, 1, 100), (600000, 8, 1, 700)):
        held = ops.selective_scan_carry_floats(most, seqs, C, N)
        for rows in sorted({1, 31, 32, 33, 64, most, *(min(most, max(1, (1 << b) // C + d)) for b in (19, 23, 25) for d in (-1, 0, 1))}):
            assert held >= ops.selective_scan_carry_floats(rows, seqs, C, N)
            for dtype in (torch.bfloat16, torch.float32):
                assert held >= (rows // ops.scan_piece(rows, C, dtype) + seqs + 1) * C * (N + 1), (C, rows)
