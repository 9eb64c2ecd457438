"""The remap's two kernels in columns of few levels, on both sides of the rule that
chooses between them (864 elements: 4 fields are split, 9 are not, 5 are not below
12 levels): each against the oracle after two steps, at ten times the one-step
bar, and the state that both remap bit for bit."""
import numpy as np
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from parity import compare, fmt

pytestmark = pytest.mark.gpu


def step(prob):
    o = oracle.OracleSession(prob)
    o.run(2)
    ref = o.state()
    o.close()
    with HipSession(prob) as h:
        h.run(2)
        out = h.state()
    rep = compare(out, ref)
    print(prob.nlev, prob.qsize, prob.params.rsplit, fmt(rep), flush=True)
    for k, (e, _) in rep.items():
        assert e <= 1e-12, (prob.nlev, prob.qsize, k, e)
    return out


@pytest.mark.parametrize("alg", [1, 2])
@pytest.mark.parametrize("nlev", [3, 4, 5, 8, 11, 12, 15, 16, 19])
def test_split_and_one_lane(nlev, alg):
    out = [step(build_problem(ne=12, nlev=nlev, qsize=q, seed=nlev, dt=100.0, remap_alg=alg)) for q in (1, 2, 6)]
    for k in ("v", "T", "dp3d", "ps_v"):
        for o in out[1:]:
            assert np.array_equal(o[k], out[0][k]), k


# tracers only: 4 are split, 5 not
@pytest.mark.parametrize("qsize", [4, 5])
@pytest.mark.parametrize("nlev", [3, 7, 11])
def test_eulerian_tracers(nlev, qsize):
    step(build_problem(ne=12, nlev=nlev, qsize=qsize, seed=nlev, dt=100.0, rsplit=0))
