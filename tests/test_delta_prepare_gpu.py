"""What the delta rule's recurrence reads of a row (csrc/hip/delta_rule.hip), at numbers of rows, heads and ranks around what its workgroups take."""
import numpy as np
import pytest
import torch

import plain_kasuvik as plain
from test_kasuvik_gpu import dev

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("heads,d,rank", [(1, 3, 1), (1, 64, 64), (2, 48, 20), (3, 64, 15), (9, 20, 16), (4, 70, 16), (5, 128, 33), (33, 16, 256), (8, 64, 64)])
def test_rows_alone_and_eight_at_a_time(heads, d, rank):
    from kvcm_amd import ops
    rng, D, T = np.random.default_rng(d + rank), heads * d, 4101
    p = rng.normal(size=(T, 2 * D + rank))
    ab, w0, w2 = rng.normal(size=D), rng.normal(size=D), rng.normal(size=(D, rank)) / np.sqrt(rank)
    proj, out = dev(p), {}
    for rows in (1, 7, 500, T):
        o = [torch.full((rows, D), float("nan"), device=DEV) for _ in range(3)]
        ops.delta_prepare(proj[:rows, :D], proj[:rows, D:2 * D], dev(ab), proj[:rows, 2 * D:], dev(w2.T.copy()), dev(w0), *o, heads, d, rows)
        out[rows] = o
    for rows, o in out.items():      # a row's bits do not depend on the rows beside it
        assert all(torch.equal(x, y[:rows]) for x, y in zip(o, out[T]))
    k = p[:, :D].reshape(T, heads, d)
    u = (k / np.sqrt((k ** 2).sum(-1, keepdims=True) + 1e-6)).reshape(T, D)
    want = (np.exp(-np.exp(-0.5) * plain.sigmoid(np.tanh(p[:, 2 * D:]) @ w2.T + w0)), plain.sigmoid(p[:, D:2 * D] + ab) * u, u)
    # values of up to one: sums of up to 256 products of up to a few, and some roundings each
    for got, ref in zip(out[T], want):
        np.testing.assert_allclose(got.double().cpu().numpy(), ref, rtol=0, atol=4e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [1, 16])
def test_as_many_heads_as_rows(rank):
    """More heads than a launch's second and third dimensions take: a channel each, whose u is its key's sign."""
    from kvcm_amd import ops
    heads, rows = 4 * 65535 + 5, 2
    g = torch.Generator(device=DEV).manual_seed(rank)
    k, a = (torch.randn(rows, heads, generator=g, device=DEV) + 2 for _ in range(2))
    w2, low = torch.randn(rank, heads, generator=g, device=DEV), torch.randn(rows, rank, generator=g, device=DEV)
    zero, o = torch.zeros(heads, device=DEV), [torch.full((rows, heads), float("nan"), device=DEV) for _ in range(3)]
    ops.delta_prepare(k, a, zero, low, w2, zero, *o, heads, 1, rows)
    u = k.double() / torch.sqrt(k.double() ** 2 + 1e-6)
    want = torch.exp(-np.exp(-0.5) * torch.sigmoid(torch.tanh(low.double()) @ w2.double())), torch.sigmoid(a.double()) * u, u
    for got, ref in zip(o, want):
        assert float((got.double() - ref).abs().max()) < 4e-6      # as above
