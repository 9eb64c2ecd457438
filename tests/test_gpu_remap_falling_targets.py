"""Columns whose surface pressure fell so far that a target thickness is negative:
a target interface then lies above the one before.  The kernel that splits columns
over lane groups remaps them as the one with a lane a column does (whose search
for a target goes on from the last one's cell), bit for bit: the same state with
few tracers (split) and with many (one lane a column)."""
import numpy as np
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from test_gpu_remap_paths import kids

pytestmark = pytest.mark.gpu


def falling(nlev, qsize, layer):
    """A layer of 0.05 Pa at the initial pressure that holds 0.3 of ps"""
    prob = build_problem(ne=10, nlev=nlev, qsize=qsize, seed=4, u_perturb=5.0)
    vc, s = prob.vcoord, prob.state
    vc.hybi[layer + 1] = vc.hybi[layer] + 0.3
    vc.hyai[layer + 1] = vc.hyai[layer] - 0.3 + 0.05 / vc.ps0
    dp = vc.dp3d(s["ps_v"][:, 0])
    s["dp3d"][:] = dp[:, None]
    s["Qdp"][:] = (s["Q"] * dp[:, None])[:, None]
    return prob


# 600 elements: 4 and 15 fields are split (one and two a wave), 11 and 27 not
@pytest.mark.parametrize("nlev,few,many,layer", [(20, 1, 8, 9), (66, 12, 24, 45)])
def test_split_columns_follow_one_lane(nlev, few, many, layer):
    prob = falling(nlev, few, layer)
    # thicknesses before the remap, and the cells of each target by itself
    o = oracle.OracleSession(prob)
    oracle.lib().oracle_debug_stop(o.h, 5)
    o.run(1)
    src = o.state()["dp3d"][:, prob.time_level[2] - 1]
    oracle.lib().oracle_debug_stop(o.h, 0)
    o.close()
    vc = prob.vcoord
    tgt = vc.dp3d(vc.hyai[0] * vc.ps0 + src.sum(1))
    cols = lambda a: np.moveaxis(a, 1, -1).reshape(-1, nlev)
    kid = kids(cols(src), cols(tgt))
    fall = (np.diff(kid, axis=1) < 0).any(1).reshape(-1, 16).any(1)
    deep = (kid > np.arange(nlev) + 1).any(1).reshape(-1, 16).any(1)
    print(nlev, "elements with falling targets: %d deep, %d not" % ((fall & deep).sum(), (fall & ~deep).sum()), flush=True)
    assert (src > 0).all() and (fall & deep).any() and (fall & ~deep).any()
    out = []
    for q in (few, many):
        with HipSession(falling(nlev, q, layer)) as h:
            h.run(1)
            out.append(h.state())
    for k in ("v", "T", "dp3d", "ps_v"):
        assert np.array_equal(out[0][k], out[1][k]), k
