"""The copies between the Fortran arrays and the device, through pinned pieces of
2 MB on up to four threads: what goes in comes back bit for bit, with arrays of
less than a piece, of several (a piece then ends inside an element's rows), with
tracer slots beyond qsize, and one element row larger than a piece."""
import numpy as np
import pytest

from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne,nlev,qsize,qsize_d", [(2, 3, 1, 1), (2, 26, 0, 1), (3, 37, 2, 5), (8, 73, 3, 3),
                                                   (8, 72, 5, 6), (2, 256, 70, 71)])
def test_round_trip(ne, nlev, qsize, qsize_d):
    prob = build_problem(ne=ne, nlev=nlev, qsize=qsize, qsize_d=qsize_d, seed=nlev)
    rng = np.random.default_rng(ne)
    for k in ("v", "T", "dp3d", "Qdp", "ps_v"):  # every value its own
        prob.state[k] = rng.uniform(1.0, 2.0, prob.state[k].shape)
    with HipSession(prob) as h:
        out = h.state()
    for k in ("v", "T", "dp3d", "Qdp", "ps_v"):
        assert np.array_equal(out[k], prob.state[k]), k
