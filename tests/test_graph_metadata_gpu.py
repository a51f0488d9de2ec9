"""Replayed decode steps whose metadata the graph fetches itself, and those whose metadata is more than it fetches (many rows, long page
tables): tokens as of steps that are launched one by one, padded rows and sampled ones included."""
import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,longest", [(1, 5), (5, 40), (49, 60), (49, 4100)])      # padded to 1, 8, 64, 64 rows; 64 x 1,024 pages at the last
def test_graphs_fetch_their_metadata(tmp_path, rows, longest):
    from kvcm_amd import Engine, EngineConfig
    d = str(tmp_path / "m")
    H.make_model_dir(d, H.TINY_D, H.WEIGHT_SEED["D"], torch.bfloat16, sharpen=H.SHARPEN["D"])
    rng = np.random.default_rng(rows + longest)
    prompts = [rng.integers(0, H.TINY_D["vocab_size"], size=longest if i == rows // 2 else 3 + i % 7).tolist() for i in range(rows)]
    out = []
    for graphs in (True, False):
        eng = Engine(d, EngineConfig(dtype="bfloat16", block_size=8, num_blocks=1024, max_seq_len=8192, max_num_seqs=64, max_batched_tokens=8192,
                                     beyond_max_position=True, use_graphs=graphs, use_programs=graphs))
        out.append(eng.generate(prompts, 6) + eng.generate(prompts[::-1], 5, temperature=0.7))      # the shape again, other metadata
        if graphs:
            assert eng.decode_graphs.graph_shapes(), "no graph was captured"
    assert out[0] == out[1]


def test_a_graph_that_fetches_less_than_a_step_holds_is_an_error(tmp_path):
    """The graph fetches what the step it was recorded from holds, not a guess at it: a step that holds more is not run."""
    from kvcm_amd import Engine, EngineConfig, ops
    d = str(tmp_path / "m")
    H.make_model_dir(d, H.TINY_D, H.WEIGHT_SEED["D"], torch.bfloat16, sharpen=H.SHARPEN["D"])
    eng = Engine(d, EngineConfig(dtype="bfloat16", block_size=8, num_blocks=64, max_seq_len=64, max_num_seqs=4, max_batched_tokens=64))
    build = eng.core.build_batch_from_plan

    def short(*args, **kw):
        layout = build(*args, **kw)
        layout.total -= 4
        return layout

    eng.core.build_batch_from_plan = short
    with pytest.raises(ops.KernelError, match="metadata of"):
        eng.generate([[1, 2, 3]], 6)
