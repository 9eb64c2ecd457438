"""The remap's kernels against the oracle: a wave per field or per pair of
fields (short columns, few fields or few elements) and one lane per column
(long columns here), with a field count for every slot layout, and columns in
which an interface rises by more than a layer."""
import numpy as np
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from parity import compare, fmt

pytestmark = pytest.mark.gpu

TOL = 1e-12  # two steps: ten times the one-step bar


def check(prob, steps=2):
    o = oracle.OracleSession(prob)
    o.run(steps)
    ref = o.state()
    o.close()
    with HipSession(prob) as h:
        h.run(steps)
        out = h.state()
    rep = compare(out, ref)
    print(prob.nlev, prob.qsize, fmt(rep), flush=True)
    for k, (e, _) in rep.items():
        assert e <= TOL, (prob.nlev, prob.qsize, k, e)


# split columns: 3 to 12 fields one a wave, 13 and more two a wave (odd counts
# leave a slot empty), 17 and more in several rounds
@pytest.mark.parametrize("nlev", [26, 33, 72, 73, 80])
@pytest.mark.parametrize("qsize", [0, 1, 9, 10, 13, 14, 30])
def test_split_columns(nlev, qsize):
    fields = None if qsize else 0
    prob = build_problem(ne=2, nlev=nlev, qsize=qsize, seed=nlev + qsize, remap_alg=1 + qsize % 2)
    if fields is None:
        check(prob)
    else:
        o = oracle.OracleSession(prob)
        o.run(2)
        ref = o.state()
        o.close()
        with HipSession(prob) as h:
            h.run(2)
            rep = compare(h.state(), ref, ("v", "T", "dp3d", "ps_v", "omega_p"))
        for k, (e, _) in rep.items():
            assert e <= TOL, (k, e)


# one lane a column: 1 to 4 fields a lane, 65 fields in a second block
@pytest.mark.parametrize("qsize", [2, 17, 40, 62])
@pytest.mark.parametrize("nlev", [81, 90])
def test_one_lane_columns(nlev, qsize):
    check(build_problem(ne=2, nlev=nlev, qsize=qsize, seed=nlev))


@pytest.mark.parametrize("rsplit", [0, 1])
def test_eulerian_tracers(rsplit):
    check(build_problem(ne=2, nlev=40, qsize=14, seed=9, rsplit=rsplit))


def kids(src, tgt):
    """The source cell of each target's lower interface, by the reference's
    search, for columns (ncol, nlev)"""
    n, nlev = src.shape
    pio = np.concatenate([np.zeros((n, 1)), np.cumsum(src, 1)], 1)
    pin = np.concatenate([np.cumsum(tgt, 1)[:, :-1], pio[:, -1:]], 1)
    out = np.zeros((n, nlev), int)
    for c in range(n):
        for k in range(nlev):
            s = k
            while s <= nlev and pio[c, s] <= pin[c, k]:
                s += 1
            out[c, k] = min(s, nlev) - 1
    return out


@pytest.mark.parametrize("qsize", [2, 14])
def test_interfaces_that_rise_by_more_than_a_layer(qsize):
    """Three layers of 1 mPa: their interfaces move by many layers in a step"""
    prob = build_problem(ne=2, nlev=20, qsize=qsize, seed=4, u_perturb=5.0)
    vc = prob.vcoord
    for k in (9, 10, 11):  # interfaces k+1 just below interface k
        vc.hyai[k + 1] = vc.hyai[9] + 1e-8 * (k - 8)
        vc.hybi[k + 1] = vc.hybi[9]
    s = prob.state
    dp = vc.dp3d(s["ps_v"][:, 0])
    s["dp3d"][:] = dp[:, None]
    s["Qdp"][:] = (s["Q"] * dp[:, None])[:, None]
    # thicknesses before the remap, and the cells its targets fall into
    o = oracle.OracleSession(prob)
    oracle.lib().oracle_debug_stop(o.h, 5)
    o.run(1)
    src = o.state()["dp3d"][:, prob.time_level[2] - 1]
    oracle.lib().oracle_debug_stop(o.h, 0)
    o.close()
    ps = vc.hyai[0] * vc.ps0 + src.sum(1)
    cols = lambda a: np.moveaxis(a, 1, -1).reshape(-1, prob.nlev)
    kid = kids(cols(src), cols(vc.dp3d(ps)))
    assert (kid > np.arange(prob.nlev) + 1).any()
    check(prob, steps=1)
