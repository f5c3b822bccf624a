"""How many workgroups share the keys of a prompt step's tiles (kernels/window_attn.py: span_shares): steps whose best count was measured, and
the sums that the rule works on."""
import numpy as np
import pytest

from swiftllm_amd.worker.batch_plan import StepEntry, plan_step
from swiftllm_amd.worker.kernels.window_attn import StepTiles, span_shares


def _shares(parts, H, G, dim, vdim, window=0):
    """parts: (keys before, tokens) of every portion."""
    plan = plan_step([StepEntry(i, np.zeros(n, dtype=np.int64), a) for i, (a, n) in enumerate(parts)])
    tiles = StepTiles(None, None, None, max(plan.target_lens_list), None, (plan.target_lens_list, plan.seq_cnt))
    row_keys, lone_keys = tiles.keys(plan.num_tokens)
    assert row_keys == int((plan.tok_pos.astype(np.int64) + 1).sum())
    assert lone_keys == sum(a + n for a, n in parts if n < 8)
    return span_shares(plan.num_tokens, plan.chunk_row0.size, H, G, dim, vdim, window, tiles.longest, row_keys, lone_keys)


@pytest.mark.parametrize("parts,narrow,wide", [
    ([(0, 2000)], (1,), (2,)), ([(0, 200)] * 8, (1,), (1,)), ([(0, 1500)] * 2, (1,), (1,)), ([(0, 500)], (1,), (4, 8)),
    # one sequence's walk is far longer than what a CU has to do in all
    ([(0, 500)] * 4 + [(8000, 1)] * 8, (4,), (4,)), ([(0, 2000)] + [(3900, 1)] * 30, (2, 4), (2, 4)), ([(0, 1000), (3900, 1)], (4,), (4, 8)),
    ([(0, 500)] + [(800, 1)] * 30, (1, 2), (2, 4)), ([(0, 200)] * 8 + [(2000, 1)], (2, 4), (4,)), ([(3500, 500)], (4, 8), (4, 8)),
    ([(0, 4000)] + [(3900, 1)] * 30, (1,), (1,)), ([(0, 1000)] * 8 + [(8000, 1)], (4,), (2, 4)),
])
def test_shares_of_measured_steps(parts, narrow, wide):
    assert _shares(parts, 8, 2, 128, 128) in narrow
    assert _shares(parts, 8, 1, 576, 512) in wide


def test_a_window_bounds_the_walk():
    parts = [(0, 2000)] + [(7000, 1)] * 4
    assert _shares(parts, 8, 2, 128, 128) == 4 and _shares(parts, 8, 2, 128, 128, window=256) == 1
    assert _shares([(0, 2000)] * 4, 8, 1, 576, 512, window=1024) == 1


def test_without_lengths_every_token_counts_as_the_longest():
    tiles = StepTiles(None, None, None, 100)
    assert tiles.keys(7) == (700, 0) and StepTiles(None, None).keys(5) == (0, 0)
    assert span_shares(7, 7, 8, 2, 128, 128, 0, 0, 0, 0) == 1
