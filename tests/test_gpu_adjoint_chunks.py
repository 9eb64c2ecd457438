"""The remap adjoint's lanes own eight scratch entries of a column each (nlev + 4
entries): level counts around whole chunks and the smallest columns, both
boundary treatments, against the PyTorch reference's gradient on the CPU (the
bar of the other adjoint cases)."""
import pytest
import torch

from hommexx_amd.adjoint import (DiffSession, energy_mismatch, initial_state, region_weight, synthetic_target,
                                 trajectory)
from hommexx_amd.problem import build_problem
from parity import rel_l2
from torch_ref import TorchStep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg", [1, 2])
@pytest.mark.parametrize("nlev", [4, 5, 11, 12, 13, 14, 19, 20, 21, 22, 28, 37])
def test_remap_adjoint_chunks(nlev, alg):
    prob = build_problem(ne=2, nlev=nlev, qsize=1, seed=nlev, rsplit=1, remap_alg=alg, t_noise=0.1)
    x0 = [a.clone().requires_grad_() for a in initial_state(prob, "cpu")]
    out = TorchStep(prob).run(*x0, 2)
    Jr = energy_mismatch(prob, *out, synthetic_target(prob, 2, "cpu"), region_weight(prob, device="cpu"))
    gref = torch.autograd.grad(Jr, x0)
    with DiffSession(prob) as s:
        x = [a.clone().requires_grad_() for a in initial_state(prob)]
        J = energy_mismatch(prob, *trajectory(s, *x, 2, 2), synthetic_target(prob, 2), region_weight(prob))
        g = torch.autograd.grad(J, x)
    for a, b, n in zip(g, gref, ("v", "T", "ps")):
        e = rel_l2(a.cpu().numpy(), b.numpy())
        print(nlev, alg, "grad %-2s rel L2 %.2e" % (n, e), flush=True)
        assert e <= 1e-9, (n, e)
