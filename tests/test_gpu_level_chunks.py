"""The dynamics kernels hold a point's levels in chunks of four or six; the
level counts here leave every kind of last chunk (full, partial, one level),
sit on both sides of the lines where the chunk length changes, and reach the
smallest and largest block.  Two steps against the oracle at ten times the
one-step bar, as the other option cases."""
import pytest

import oracle
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem
from parity import compare, fmt

pytestmark = pytest.mark.gpu


def check(prob, tol, form="fp64", fields=None, steps=2):
    o = oracle.OracleSession(prob)
    o.run(steps)
    ref = o.state()
    o.close()
    with HipSession(prob, form=form) as h:
        h.run(steps)
        out = h.state()
    rep = compare(out, ref, *([fields] if fields else []))
    print(prob.nlev, form, fmt(rep), flush=True)
    for k, (e, _) in rep.items():
        assert e <= tol, (prob.nlev, form, k, e)


@pytest.mark.parametrize("nlev", [3, 4, 5, 7, 16, 17, 63, 64, 65, 67, 71, 79, 94, 96, 97, 130])
def test_chunk_lengths(nlev):
    check(build_problem(ne=2, nlev=nlev, qsize=1, seed=nlev), 1e-12)


@pytest.mark.parametrize("over", [dict(rsplit=0), dict(moisture=True), dict(nu_div=2.5e16), dict(nu_top=0.0),
                                  dict(rsplit=2, qsplit=2)])
@pytest.mark.parametrize("nlev", [66, 70])
def test_six_level_options(nlev, over):
    check(build_problem(ne=2, nlev=nlev, qsize=2, seed=nlev, **over), 1e-12)


@pytest.mark.parametrize("nlev,nu_div", [(26, 1e16), (26, 2.5e16), (70, 1e16), (70, 2.5e16)])
def test_mixed_form(nlev, nu_div):
    # the form's bar for every prognostic field
    check(build_problem(ne=2, nlev=nlev, qsize=2, seed=nlev, nu_div=nu_div), 1e-6, form="mixed",
          fields=("v", "T", "dp3d", "ps_v", "Qdp", "Q"))
