"""Eulerian levels (rsplit == 0) at the level counts that take other kernels than
the common ones: the remap of tracers alone with one lane a column (above 80
levels), dynamics blocks of more than 512 lanes (above 128 levels, a form of its
own) and of more than 64 KB of LDS (above 170), up to the most levels.  Two steps
against the oracle at ten times the one-step bar, as the other option cases."""
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from parity import compare, fmt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("moist", [False, True])
@pytest.mark.parametrize("nlev", [81, 90, 128, 129, 171, 255, 256])
def test_eulerian_levels(nlev, moist):
    prob = build_problem(ne=2, nlev=nlev, qsize=2, seed=nlev, rsplit=0, moisture=moist)
    o = oracle.OracleSession(prob)
    o.run(2)
    ref = o.state()
    o.close()
    with HipSession(prob) as h:
        h.run(2)
        rep = compare(h.state(), ref)
    print(nlev, moist, fmt(rep), flush=True)
    for k, (e, _) in rep.items():
        assert e <= 1e-12, (nlev, moist, k, e)
