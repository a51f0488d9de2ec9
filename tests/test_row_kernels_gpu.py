"""Row kernels at the sizes where their forms change."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H", [4, 8, 12, 256, 260, 264, 2048, 2056, 4104])      # (pieces beyond 256)
def test_embedding_by_pieces_gathers_rows(H, dtype):
    from kvcm_amd import ops
    V = 37
    table = torch.randn(V + 1, H, device=DEV).to(dtype)
    ids = torch.tensor([0, V - 1, 5, -1, V, 5, 17], dtype=torch.int32, device=DEV)      # (ids without a row give zeros)
    known = (ids >= 0) & (ids < V)
    for rows in (table[:V], table.flatten()[1:1 + V * H].view(V, H)):      # rows that begin at any entry go entry by entry
        out = torch.full((len(ids), H), float("nan"), device=DEV)
        ops.embed(ids, rows, out)
        want = rows[ids.clamp(0, V - 1).long()].float() * known[:, None]
        assert torch.equal(out, want)
