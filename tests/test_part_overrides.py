"""Parts derived from this package's own that replace a method: the arrangement runs the replacement, whatever shorter way it has for the base
(no GPU)."""
from types import SimpleNamespace

import pytest
import torch

from kvcm_amd.parts import llama_parts
from kvcm_amd.parts.base import Mixer, Norm, said_with
from kvcm_amd.parts.chain_norm_parts import GatedFeedForward
from kvcm_amd.parts.conv_attention_parts import ConvWindowPoolAttention, ParallelMixers
from kvcm_amd.parts.llama_parts import GQAAttention, PreNormResidual, RMSNorm, Rotary, SwiGLU
from kvcm_amd.parts.recurrent_parts import SelectiveScanMixer
from kvcm_amd.parts.routed_parts import RoutedExperts


class _Fold(Norm):
    """A norm that folds: adds what it is given and hands the rows on."""
    defers = accepts_partial_sums = True

    def __init__(self):
        pass

    def forward(self, x, out, add=None, rows=None, defer=False):
        return x + (0 if add is None else add)


def _bare(cls, **attributes):
    part = object.__new__(cls)
    vars(part).update(attributes)
    return part


STEP = SimpleNamespace(rows=2, fold_norms=True, ws=lambda name, shape, dtype=None: torch.zeros(shape, dtype=dtype))


def test_a_block_runs_mixers_and_feed_forwards_with_a_forward_of_their_own():
    class Double(GQAAttention):
        def forward(self, step, h):
            return 2 * h

    class Triple(SwiGLU):
        def forward(self, step, h):
            return 3 * h

    class Late(Double):
        defers = True

        def forward(self, step, h, defer=False):
            return 5 * h if defer else None

    x = torch.ones(2, 4)
    for mixer, result in ((_bare(Double), 3 * (1 + 2)), (_bare(Late), 3 * (1 + 5)),
                          (_bare(GQAAttention, forward=lambda step, h: 2 * h), 3 * (1 + 2))):      # an instance's own, as a wrapper leaves it
        block = _bare(PreNormResidual, parts=dict(norm_mixer=_Fold(), norm_ffn=_Fold(), mixer=mixer, ffn=_bare(Triple)))
        assert torch.equal(block.forward(STEP, x, None), torch.full((2, 4), float(result)))
    block = _bare(PreNormResidual, parts=dict(norm_mixer=_Fold(), norm_ffn=_Fold(), mixer=_bare(Double), ffn=_bare(SwiGLU, forward=lambda step, h: h)))
    assert torch.equal(block.forward(STEP, x, None), torch.full((2, 4), 3.0))


def test_a_forward_of_its_own_gets_normed_rows_and_not_rows_to_norm():
    """32-bit rows that a product norms itself go to the package's own forwards only, or to those that say they take them."""
    class RowsToNorm:
        def __init__(self, x, weight, eps, out):
            self.x = x

    ops = SimpleNamespace(PendingProduct=type("PendingProduct", (), {}), RowsToNorm=RowsToNorm, can_norm_rows=lambda x, weight, out: True,
                          rmsnorm=lambda x, weight, out, eps, add=None, rows=None: out.copy_(x if add is None else x.add_(add)))
    norm = _bare(RMSNorm, ctx=SimpleNamespace(ops=ops), params=dict(eps=0.0), w=dict(weight=None), _folded=None)

    class Double(GQAAttention):
        def forward(self, step, h):
            return 2 * h

    class Triple(SwiGLU):
        def forward(self, step, h):
            return 3 * h

    class Takes(Triple):
        accepts_rows_to_norm = True

        def forward(self, step, h):
            return 5 * h.x

    run = lambda mixer, ffn: _bare(PreNormResidual, parts=dict(norm_mixer=norm, norm_ffn=norm, mixer=mixer, ffn=ffn)).forward(STEP, torch.ones(2, 4), None)
    assert torch.equal(run(_bare(Double), _bare(Triple)), torch.full((2, 4), 9.0))
    assert torch.equal(run(_bare(GQAAttention, forward=lambda step, h: 2 * h), _bare(SwiGLU, forward=lambda step, h: 3 * h)), torch.full((2, 4), 9.0))
    norm_two = _bare(RMSNorm, **{**vars(norm), "w": dict(weight=1)})
    got = _bare(PreNormResidual, parts=dict(norm_mixer=norm, norm_ffn=norm_two, mixer=_bare(Double, forward=lambda step, h: None), ffn=_bare(Takes))).forward(
        STEP, torch.ones(2, 4), None)
    assert torch.equal(got, torch.full((2, 4), 5.0))
    out = torch.zeros(2, 4)
    assert norm.forward(torch.ones(2, 4), out, defer=True) is out and isinstance(norm.forward(torch.ones(2, 4), out, defer="rows"), RowsToNorm)


@pytest.mark.parametrize("side", ("left", "right"))
def test_mixers_side_by_side_run_a_forward_of_their_own(side):
    class Window(ConvWindowPoolAttention):
        def forward(self, step, h):
            return 2 * h

    class Scan(SelectiveScanMixer):
        def forward(self, step, h):
            return 3 * h

    class Other(Mixer):
        buffers = {"kept": 1}      # any attribute of that name

        def __init__(self):
            pass

        def forward(self, step, h):
            return 7 * h

    h = torch.ones(2, 4)
    for part, factor in ((_bare(Window), 2), (_bare(Scan), 3), (Other(), 7)):
        other = _bare(ConvWindowPoolAttention if side == "right" and not isinstance(part, Window) else SelectiveScanMixer, forward=lambda step, h: 11 * h)
        pair = _bare(ParallelMixers, params={}, w=dict(w_left=None, w_right=None), ctx=None, **{side: part, ("left", "right")[side == "left"]: other})
        out = pair.forward(STEP, h)
        assert torch.equal(getattr(out, "ab"[side == "right"]), factor * h) and torch.equal(getattr(out, "ab"[side == "left"]), 11 * h)


def test_a_shared_feed_forward_with_a_forward_of_its_own_is_not_folded_into_the_experts():
    class Scaled(GatedFeedForward):
        def forward(self, step, h):
            return 2 * super().forward(step, h)

    h = torch.zeros(2, 64, dtype=torch.bfloat16)
    ctx = SimpleNamespace(ops=SimpleNamespace(moe_few_beside_takes=lambda *a: True))
    for shared, folds in ((_bare(GatedFeedForward, params={}, w=dict(w_gate_up=None)), True), (_bare(Scaled, params={}, w=dict(w_gate_up=None)), False),
                          (_bare(GatedFeedForward, params={}, w=dict(w_gate_up=None), forward=lambda step, h: h), False)):
        routed = _bare(RoutedExperts, gated=True, by_ends=False, shared=shared, ctx=ctx)
        assert routed._beside(h, 64, 64, 2, 8) == folds


def test_who_says_what_for_which_method():
    class Turned(Rotary):
        def apply(self, step, qkv, *args, **kw):
            return False

    class Both(Turned):
        def rotation_table(self, step, head_dim):
            return None

    assert said_with(_bare(Rotary), "rotation_table", "apply") and said_with(_bare(Both), "rotation_table", "apply")
    assert not said_with(_bare(Turned), "rotation_table", "apply")
    assert not said_with(_bare(Rotary), "nothing", "apply")
    assert all(said_with(_bare(c), "defers", "forward") for c in (GQAAttention, SwiGLU))
    assert all(said_with(_bare(c), "stages", "forward") for c in (ConvWindowPoolAttention, SelectiveScanMixer))
    assert llama_parts.said_with is said_with
