"""A last chunk that is not full does the work of a full one, no more: the
tracer stages of 25, 26 and 30 levels (whole chunks of eight: 32) take the time
that 32 levels take.  Both are the least of five; the levels that only fill the
chunk up once cost their waves five limiter iterations for one, 2.2 times the
time of 32 levels."""
import pytest

from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem

pytestmark = pytest.mark.gpu


def advection_ms(nlev, form):
    prob = build_problem(ne=12, nlev=nlev, qsize=24, seed=1)
    with HipSession(prob, form=form) as h:
        h.run(2)
        best = float("inf")
        for _ in range(5):
            h.profile_reset()
            h.profile(True, only="euler_advect")
            h.run(4)
            h.profile(False)
            best = min(best, h.profile_report()["euler_advect"][1] / 4)
    return best


@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_partial_chunk_costs_a_full_one(form):
    full = advection_ms(32, form)
    for nlev in (25, 26, 30):
        t = advection_ms(nlev, form)
        print(form, nlev, "%.3f ms, 32 levels %.3f" % (t, full), flush=True)
        assert t <= 1.3 * full, (form, nlev, t, full)
