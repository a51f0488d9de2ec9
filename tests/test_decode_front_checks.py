"""What the attention half in one launch refuses before anything is launched (no GPU: tensors without memory)."""
import pytest
import torch

from kvcm_amd import ops

NH, NKV, HD, B, H, M = 4, 2, 64, 32, 256, 2
BF = torch.bfloat16


def _pending(kcache, vcache, launched):
    e = lambda *shape, dtype=torch.int32: torch.empty(shape, dtype=dtype, device="meta")
    p = ops.PendingAttention(None, e(M, H, dtype=BF), e((NH + 2 * NKV) * HD, H, dtype=BF), e(M, NH * HD, dtype=BF), e(H, NH * HD, dtype=BF), e(M, H, dtype=BF), None,
                             (kcache, vcache), e(M, 4), 4, e(M), e(M), e(M), None, (NH, NKV, HD), 0.125, 1, lambda: launched)
    return p.run_with_norm(e(M, H, dtype=torch.float32), e(H, dtype=BF), 1e-5, e(8, H, dtype=BF), e(8, H // 8, dtype=torch.float32), None)


@pytest.mark.parametrize("pages", (2 ** 35 // (NKV * B * HD) + 1, 2 ** 35 // (NKV * B * HD)))
def test_caches_beyond_its_offsets_are_refused(monkeypatch, pages):
    """It keeps a token's place in a layer's cache as 32 bits in units of 8 elements, as the decode kernel does that it runs in place of."""
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    kc, vc = torch.empty(pages, NKV, B, HD, dtype=BF, device="meta"), torch.empty(pages, NKV, HD, B, dtype=BF, device="meta")
    if kc.numel() > 2 ** 35:
        with pytest.raises(ValueError, match="page offsets"):
            _pending(kc, vc, None)
    else:      # as far as the hand-over buffers
        with pytest.raises(TypeError):
            _pending(kc, vc, None)


def test_caches_of_different_pages_are_refused(monkeypatch):
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    with pytest.raises(ValueError, match="value cache"):
        _pending(torch.empty(9, NKV, B, HD, dtype=BF, device="meta"), torch.empty(8, NKV, HD, B, dtype=BF, device="meta"), None)
