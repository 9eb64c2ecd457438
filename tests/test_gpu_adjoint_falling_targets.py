"""The adjoint of the remap where target interfaces fall (a target thickness is
negative): each target's source cell is the one that the forward remap takes, whose
search goes on from the last target's cell.  Against central differences of the
forward step, in the columns concerned.

The thin layer there (0.05 Pa) sets the tolerance: a difference moves its interfaces
by 1e-5 to 1e-3 Pa, which truncates at (1e-3/0.05)^2 = 4e-4 of the terms that hold
it and rounds at 1e-11/1e-5 = 1e-6; outputs of the layer itself and its neighbours,
divided by such thicknesses, are left out.  1e-3 of the derivative; with each target
searched by itself it was off by 0.3 to 1.5."""
import numpy as np
import pytest
import torch

import oracle
from hommexx_amd.adjoint import DiffSession
from test_gpu_remap_falling_targets import falling
from test_gpu_remap_paths import kids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg", [1, 2])
def test_adjoint_is_the_derivative(alg):
    nlev, layer = 20, 9
    prob = falling(nlev, 1, layer)
    prob.params.remap_alg = alg
    # thicknesses before the remap, and the cells of each target by itself
    o = oracle.OracleSession(prob)
    oracle.lib().oracle_debug_stop(o.h, 5)
    o.run(1)
    src = o.state()["dp3d"][:, prob.time_level[2] - 1]
    oracle.lib().oracle_debug_stop(o.h, 0)
    o.close()
    vc = prob.vcoord
    cols = lambda a: np.moveaxis(a, 1, -1).reshape(-1, nlev)
    kid = kids(cols(src), cols(vc.dp3d(vc.hyai[0] * vc.ps0 + src.sum(1))))
    fall = (np.diff(kid, axis=1) < 0).any(1)
    assert fall.any()
    where = torch.as_tensor(fall.reshape(-1, 4, 4), dtype=torch.float64, device="cuda")
    with DiffSession(prob) as s:
        x = s.get_state()
        g = torch.Generator(device="cuda").manual_seed(1)
        draw = lambda a: torch.randn(a.shape, generator=g, dtype=torch.float64, device="cuda")
        lam = [draw(x[0]) * where[:, None, None], draw(x[1]) * where[:, None], torch.zeros_like(x[2])]
        for a in lam[:2]:
            a[:, layer - 1:layer + 3] = 0
        grad = [a.clone() for a in lam]
        s.adjoint_step(x, grad)
        for i, step in ((0, 1e-7), (1, 1e-7), (2, 1e-9)):
            d = draw(x[i]) * x[i].abs().mean()
            y = []
            for e in (step, -step):
                z = [a.clone() for a in x]
                z[i] += e * d
                s.dynamics_step(z)
                y.append(z)
            fd = sum(float((l * (p - q)).sum()) for l, p, q in zip(lam, *y)) / (2 * step)
            ad = float((grad[i] * d).sum())
            print(alg, "v T ps".split()[i], "adjoint %.9e, differences %.9e" % (ad, fd), flush=True)
            assert abs(ad - fd) <= 1e-3 * abs(fd)
