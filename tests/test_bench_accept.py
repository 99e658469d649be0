"""bench.py's CPU accept step: the drafts are drawn, so a nucleus that leaves out the first ids is no error."""
import os
import sys

import numpy as np
import pytest

import oracle as O

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("top_p", [1.0, 0.95])
def test_port_accept_step_draws_its_drafts(top_p):
    rng = np.random.default_rng(2)
    k, V = 3, 4096
    target = (rng.standard_normal((k + 1, V)) * 2.5).astype(np.float32)
    draft = (target[:k] + rng.standard_normal((k, V)) * 0.5).astype(np.float32)
    target[:, :k], draft[:, :k] = -9.0, -9.0  # ids 0 .. 2 are outside q's nucleus
    if top_p < 1.0:
        with pytest.raises(ValueError):
            O.accept_logits(target, draft, np.arange(k, dtype=np.int32), 1.0, top_p, 5, 0)
    for step in range(8):
        d, got = bench.port_accept_step(target, draft, 1.0, top_p, 5, step)
        assert d.tolist() == [O.sample_v2(O.probabilities(draft[j], 1.0, top_p), 5, step, j, bench.DRAFT) for j in range(k)]
        assert got.as_tuple() == O.accept_logits(target, draft, d, 1.0, top_p, 5, step).as_tuple()
