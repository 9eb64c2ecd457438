"""Copies of arrays that fit one pinned buffer together (2 MB) go through it side by
side: what goes in comes back bit for bit on both sides of that line (24 elements
and one tracer: 48 and 49 levels in, 42 and 43 levels out), with a tracer slot
beyond qsize."""
import numpy as np
import pytest

from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlev", [3, 42, 43, 48, 49])
def test_round_trip(nlev):
    prob = build_problem(ne=2, nlev=nlev, qsize=1, qsize_d=2, seed=nlev)
    rng = np.random.default_rng(nlev)
    fields = ("v", "T", "dp3d", "Qdp", "ps_v")
    for k in fields:  # every value its own
        prob.state[k] = rng.uniform(1.0, 2.0, prob.state[k].shape)
    with HipSession(prob) as h:
        for _ in range(2):  # (the buffer is kept)
            out = h.state()
            for k in fields:
                assert np.array_equal(out[k], prob.state[k]), k
