"""The tracer kernels hold an element's levels in chunks of eight, two to a lane:
level counts that leave one to eight levels in the last chunk, tracer counts
down to none or one (the prefetch then re-reads the last), both limiters and the
three forms of the biharmonic; a larger grid whose tracers one to several
blocks share.  Two steps against the oracle at ten times the
one-step bar; the mixed form at its own bar."""
import numpy as np
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from parity import compare, fmt

pytestmark = pytest.mark.gpu

TRACERS = ("v", "T", "dp3d", "ps_v", "Qdp", "Q")


def tensor(prob, seed):
    rng = np.random.default_rng(seed)
    tv = np.zeros((prob.nelem, 2, 2, 4, 4))
    tv[:, 0, 0], tv[:, 1, 1] = rng.uniform(0.5, 1.5, (2, prob.nelem, 4, 4))
    tv[:, 0, 1] = tv[:, 1, 0] = rng.uniform(-0.3, 0.3, (prob.nelem, 4, 4))
    prob.metric["tensorvisc"] = tv


def check(prob, tol, form="fp64", fields=None):
    o = oracle.OracleSession(prob)
    o.run(2)
    ref = o.state()
    o.close()
    with HipSession(prob, form=form) as h:
        h.run(2)
        rep = compare(h.state(), ref, *([fields] if fields else []))
    print(prob.nlev, prob.qsize, form, fmt(rep), flush=True)
    for k, (e, _) in rep.items():
        assert e <= tol, (prob.nlev, prob.qsize, form, k, e)


@pytest.mark.parametrize("limiter", [8, 9])
@pytest.mark.parametrize("nlev,qsize", [(8, 1), (9, 5), (10, 2), (15, 3), (23, 9), (24, 1), (31, 4)])
def test_last_chunk(nlev, qsize, limiter):
    check(build_problem(ne=2, nlev=nlev, qsize=qsize, seed=nlev, limiter_option=limiter), 1e-12)


# ne=6: 216 elements; the tracers run in one, two, three (uneven) or more shares
@pytest.mark.parametrize("nlev,qsize", [(72, 3), (40, 5), (20, 7), (16, 7), (9, 11)])
def test_tracer_shares(nlev, qsize):
    check(build_problem(ne=6, nlev=nlev, qsize=qsize, seed=qsize), 1e-12)


def test_no_tracers():
    check(build_problem(ne=2, nlev=17, qsize=0, seed=5), 1e-12, fields=("v", "T", "dp3d", "ps_v", "omega_p"))


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("nlev,qsize,scaling", [(17, 2, 3.2), (20, 1, 3.2), (17, 1, 0.0), (22, 6, 0.0)])
def test_biharmonic_forms(nlev, qsize, scaling, form):
    prob = build_problem(ne=2, nlev=nlev, qsize=qsize, seed=nlev, hypervis_scaling=scaling)
    if scaling:
        tensor(prob, nlev)
    if form == "mixed":
        check(prob, 1e-6, form, TRACERS)
    else:
        check(prob, 1e-12)
