"""What is timed: the preqx step as its users call it.

Four kinds of pass, each through the public entry points:

* ``step``: a user's own driver with the state on the GPU.  It hands over the
  dynamics state of a member (v, T, ps; ``hommexx_hip_set_state``), runs
  ``calls`` remap intervals (``prim_run_subcycle_c``) and takes back the
  prognostic fields (``hommexx_hip_get_state``, ``hommexx_hip_get_field``).
* ``coupled``: a Fortran-like host: forcing tendencies from host arrays
  (``f90_push_forcing_to_cxx``), the intervals of one physics step, and every
  result back into host arrays (``cxx_push_results_to_f90``).
* ``adjoint``: one call of the adjoint step (``DiffSession.adjoint_step``).
* ``gradient``: a checkpointed trajectory with its loss and the gradients
  through ``torch.autograd`` (``adjoint.trajectory``).

The library holds one simulation per process.  A prepared state is therefore
the open simulation, which all states of a case share, plus the member's own
arrays.  Preparing a state sets the simulation's tracers; a pass sets the
dynamics state and leaves the tracers where the pass before it left them, as
in a running model.

``exact`` restates the step in plain torch, in 64 bits and vectorised over
elements, levels and tracers.
"""
import ctypes
import math

import numpy as np
import torch

from hommexx_amd.adjoint import DiffSession, energy_mismatch, region_weight, synthetic_target, trajectory
from hommexx_amd.hip import HipSession
from hommexx_amd.problem import build_problem, make_forcing

DEFAULTS = {"ne": 4, "nlev": 26, "qsize": 4, "calls": 1, "form": "fp64", "rsplit": 1, "qsplit": 1, "limiter": 8,
            "alg": 1, "moist": False, "kind": "step", "every": 4}


def listed():
    return [
        # the smallest run of the tests (the default of build_problem): launches and latency
        _case("step ne4 L26 Q4", ne=4, nlev=26, qsize=4),
        # a regression-test sized run with the reference's rsplit = 3
        _case("step ne8 L72 Q4 r3", ne=8, nlev=72, qsize=4, rsplit=3, calls=2),
        # odd everything: element and level counts that fill no tile, moist physics,
        # the clip-and-sum limiter, fixed-parabola remap, two dynamics steps per tracer step
        _case("step ne11 L30 Q7 moist", ne=11, nlev=30, qsize=7, rsplit=2, qsplit=2, limiter=9, alg=2, moist=True,
              calls=2),
        # the size of the differentiable form's workload, run forward
        _case("step ne16 L72 Q4", ne=16, nlev=72, qsize=4, calls=6),
        # the benchmark: half an hour of model time at 300 s
        _case("step ne30 L72 Q40", ne=30, nlev=72, qsize=40, calls=6),
        # the same in the reference's benchmark settings (remap every third step)
        _case("step ne30 L72 Q40 r3", ne=30, nlev=72, qsize=40, rsplit=3, calls=2),
        # the benchmark in the mixed-precision form
        _case("mixed ne30 L72 Q40", ne=30, nlev=72, qsize=40, form="mixed", calls=6),
        # the largest mesh: few tracers, so the dynamics and its exchanges count
        _case("step ne60 L72 Q10", ne=60, nlev=72, qsize=10, calls=3),
        # one physics interval of a coupled host: six steps, forcing in, results out
        _case("coupled ne8 L72 Q4", kind="coupled", ne=8, nlev=72, qsize=4, calls=6),
        # the adjoint step: the smallest (Eulerian levels) and the benchmark's
        _case("adjoint ne4 L26 r0", kind="adjoint", ne=4, nlev=26, qsize=0, rsplit=0),
        _case("adjoint ne16 L72 r1", kind="adjoint", ne=16, nlev=72, qsize=4, rsplit=1),
        # a small assimilation window, forward and backward
        _case("gradient ne8 L72 r1", kind="gradient", ne=8, nlev=72, qsize=1, rsplit=1, calls=8, every=4),
    ]


def _case(name=None, **over):
    c = dict(DEFAULTS, **over)
    if name:
        c["name"] = name
    return c


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choices(("step", "coupled", "adjoint", "gradient"), (12, 2, 3, 2))[0]
    nlev = rng.choice((26, 30, 72, 72, rng.randint(20, 100)))
    if kind == "step":
        ne, qsize, calls = log(2, 48), log(1, 48), rng.randint(1, 4)
        rsplit, qsplit = rng.choice((1, 1, 2, 3)), rng.choice((1, 1, 1, 2))
        # no more work than the benchmark's six steps
        while ne * ne * nlev * (qsize + 12) * calls * rsplit * qsplit > 30 * 30 * 72 * 52 * 6:
            calls, ne = max(1, calls - 1), ne - 1
        return _case(ne=ne, nlev=nlev, qsize=qsize, calls=calls, form=rng.choice(("fp64", "fp64", "mixed")),
                     rsplit=rsplit, qsplit=qsplit, limiter=rng.choice((8, 8, 9)), alg=rng.choice((1, 1, 2)),
                     moist=rng.random() < 0.25)
    if kind == "coupled":
        return _case(kind=kind, ne=log(3, 12), nlev=nlev, qsize=log(1, 10), calls=rng.randint(2, 6),
                     rsplit=rng.choice((1, 3)))
    if kind == "adjoint":
        return _case(kind=kind, ne=log(2, 20), nlev=nlev, qsize=rng.randint(0, 4), rsplit=rng.choice((0, 1, 1, 2)),
                     alg=rng.choice((1, 2)))
    return _case(kind=kind, ne=log(2, 10), nlev=nlev, qsize=1, rsplit=rng.choice((0, 1)), calls=rng.randint(2, 8),
                 every=rng.choice((2, 4, 8)))


def work(case):
    """Bytes and operations of a pass: every call reads the prognostic fields
    and the element metric once and writes its results once.  Operations: per
    point, about 450 for a dynamics stage, 600 for a hyperviscosity subcycle,
    250 per tracer step and tracer, 120 per remapped field."""
    c, p = case, 8.0 * 16 * 6 * case["ne"] ** 2 * case["nlev"]
    q, dyn = c["qsize"], c["qsplit"] * max(c["rsplit"], 1)
    metric = 30.0 / c["nlev"]
    point = dyn * (5 * 450 + 3 * 600)
    if c["kind"] in ("step", "coupled"):
        flops = point + max(c["rsplit"], 1) * 250 * q + 120 * (3 + q)
        # in: v, T, ps, Qdp; out: v, T, dp3d, omega, Qdp, Q
        per_call = 3 + q + 5 + 2 * q + metric
        # members in and results out of a pass
        ends = (6 + 2 * q) if c["kind"] == "step" else (4 + q) + 25 + 2 * q
        return {"bytes": p * (c["calls"] * per_call + ends), "flops": p / 8 * flops * c["calls"]}
    if c["kind"] == "adjoint":  # the state in, the adjoint in and out
        return {"bytes": p * (3 + 6 + metric), "flops": p / 8 * 3 * (point + 120 * 3)}
    # trajectory: forward and backward of each call, the checkpoints, the gradients
    return {"bytes": p * (c["calls"] * (2 * (6 + metric) + 9)), "flops": p / 8 * c["calls"] * 4 * (point + 120 * 3)}


# ------------------------------------------------------------- simulation
_open = {"key": None, "sim": None}


def _problem(c):
    ne, nu = c["ne"], 1e15 * (30.0 / c["ne"]) ** 3.2
    return build_problem(ne=ne, nlev=c["nlev"], qsize=c["qsize"], seed=1, dt=300.0 * min(1.0, 30.0 / ne), nu=nu, nu_p=nu,
                         nu_q=nu, nu_s=nu, nu_div=nu, rsplit=c["rsplit"], qsplit=c["qsplit"],
                         limiter_option=c["limiter"], remap_alg=c["alg"], moisture=c["moist"],
                         ftype=0 if c["kind"] == "coupled" else -1)


def _simulation(c):
    """The open simulation of this configuration (opened if another one is)"""
    key = tuple(c[k] for k in DEFAULTS if k not in ("calls", "every"))
    if _open["key"] != key:
        if _open["sim"]:
            _open["sim"]["session"].close()
        _open.update(key=None, sim=None)
        prob = _problem(c)
        diff = c["kind"] in ("adjoint", "gradient")
        session = DiffSession(prob) if diff else HipSession(prob, form=c["form"])
        h = session.h if diff else session
        lib = h.L
        pt = ctypes.c_void_p
        lib.hommexx_hip_get_state.argtypes = lib.hommexx_hip_set_state.argtypes = [pt, pt, pt]
        lib.hommexx_hip_get_field.argtypes = [ctypes.c_int, ctypes.c_int, pt]
        s, n0 = prob.state, prob.time_level[1] - 1
        pos = torch.as_tensor(prob.mesh.pos, device="cuda")
        x, y, z = pos.unbind(-1)
        _open.update(key=key, sim={
            "session": session, "h": h, "prob": prob,
            "start": [torch.as_tensor(np.ascontiguousarray(s[k][:, n0]), device="cuda") for k in ("v", "T", "ps_v")],
            # smooth patterns, continuous over the element edges
            "basis": torch.stack([x, y, z, x * y, y * z, z * x, x * x - y * y, x * y * z]),
            "coslat": torch.sqrt(x * x + y * y),
            "qdp": np.empty_like(s["Qdp"]),
        })
    return _open["sim"]


def _ref(a):
    return ctypes.byref(ctypes.c_void_p(a.ctypes.data))


def _member(sim, seed):
    """(v, T, ps) of a member: the balanced jet plus smooth perturbations of
    about 1 m/s, 0.3 K and 1 hPa that vary from level to level"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v, T, ps = (a.clone() for a in sim["start"])
    basis, nlev = sim["basis"], T.shape[1]

    def pattern(n):
        w = torch.randn(n, len(basis), generator=g, device="cuda", dtype=torch.float64) / len(basis)
        return torch.tensordot(w, basis, 1).transpose(0, 1).contiguous()

    for i in range(2):
        v[:, :, i] += sim["coslat"][:, None] * pattern(1)
        v[:, :, i] += 0.3 * sim["coslat"][:, None] * pattern(nlev)
    T += 0.3 * pattern(nlev)
    ps += 100.0 * pattern(1)[:, 0]
    return v, T, ps


def _tracers(sim, seed):
    """Qdp of a member: the smooth tracers, each scaled by a factor of the seed"""
    base, prob = sim["prob"].state["Qdp"], sim["prob"]
    f = np.random.default_rng(seed).uniform(0.5, 1.0, base.shape[2])
    if prob.params.moisture:
        f[0] *= 0.02  # specific humidity
    torch.mul(torch.from_numpy(base), torch.from_numpy(f).view(1, 1, -1, 1, 1, 1), out=torch.from_numpy(sim["qdp"]))
    return sim["qdp"]


def _load(sim, qdp):
    """the simulation as at its start, with these tracers"""
    h, s = sim["h"], sim["prob"].state
    h.L.init_elements_states_c(_ref(s["v"]), _ref(s["T"]), _ref(s["dp3d"]), _ref(qdp), _ref(s["ps_v"]))
    h.L.init_time_level_c(*[ctypes.byref(ctypes.c_int(x)) for x in sim["prob"].time_level])
    h._check("init_elements_states_c")


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    sim = _simulation(c)
    prob = sim["prob"]
    state = {"case": c, "sim": sim, "x": _member(sim, seed)}
    if c["kind"] in ("step", "coupled"):
        _load(sim, _tracers(sim, seed))
    if c["kind"] == "coupled":
        state["forcing"] = make_forcing(prob, seed)
        s = prob.state
        state["host"] = {k: np.zeros_like(s[k]) for k in ("v", "T", "dp3d", "Qdp", "Q", "ps_v")}
        state["host"]["omega_p"] = np.zeros((prob.nelem, prob.nlev, 4, 4))
    elif c["kind"] == "adjoint":
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        state["lam"] = [torch.randn(a.shape, generator=g, dtype=torch.float64, device="cuda") for a in state["x"]]
    elif c["kind"] == "gradient":
        state["target"] = synthetic_target(prob, seed)
        state["weight"] = region_weight(prob)
    torch.cuda.synchronize()
    return state


# -------------------------------------------------------------------- passes
def run(state):
    return {"step": _run_step, "coupled": _run_coupled, "adjoint": _run_adjoint,
            "gradient": _run_gradient}[state["case"]["kind"]](state)


def _set_state(sim, x):
    torch.cuda.synchronize()  # the library works on a stream of its own
    sim["h"].L.hommexx_hip_set_state(*[a.data_ptr() for a in x])


def _run_step(state):
    c, sim = state["case"], state["sim"]
    h, x = sim["h"], state["x"]
    _set_state(sim, x)
    h.run(c["calls"])
    out = [torch.empty_like(a) for a in x]
    qdp = torch.empty((c["qsize"],) + x[1].shape, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    h.L.hommexx_hip_get_state(*[a.data_ptr() for a in out])
    for q in range(c["qsize"]):
        h.L.hommexx_hip_get_field(4, q, qdp[q].data_ptr())
    h._check("get_field")
    return {"v": out[0], "T": out[1], "ps": out[2], "qdp": qdp}


def _run_coupled(state):
    c, sim, f, o = state["case"], state["sim"], state["forcing"], state["host"]
    h = sim["h"]
    _set_state(sim, state["x"])
    dp = ctypes.POINTER(ctypes.c_double)
    h.L.f90_push_forcing_to_cxx(*[a.ctypes.data_as(dp) for a in (f["FM"], f["FT"], f["FQ"], o["Qdp"])])
    nstep, _, n0, _ = h.run(c["calls"])
    h.L.cxx_push_results_to_f90(*[_ref(o[k]) for k in ("v", "T", "dp3d", "Qdp", "Q", "ps_v", "omega_p")])
    h._check("cxx_push_results_to_f90")
    level = nstep // c["qsplit"] % 2
    return {"v": o["v"][:, n0], "T": o["T"][:, n0], "ps": o["ps_v"][:, n0], "dp3d": o["dp3d"][:, n0],
            "qdp": o["Qdp"][:, level], "Q": o["Q"], "omega_p": o["omega_p"]}


def _run_adjoint(state):
    lam = [a.clone() for a in state["lam"]]
    state["sim"]["session"].adjoint_step(state["x"], lam)
    return {"v": lam[0], "T": lam[1], "ps": lam[2]}


def _run_gradient(state):
    c, sim = state["case"], state["sim"]
    x = [a.clone().requires_grad_() for a in state["x"]]
    end = trajectory(sim["session"], *x, c["calls"], c["every"])
    loss = energy_mismatch(sim["prob"], *end, state["target"], state["weight"])
    loss.backward()
    return {"loss": loss.detach(), "v": end[0].detach(), "T": end[1].detach(), "ps": end[2].detach(),
            "gv": x[0].grad, "gT": x[1].grad, "gps": x[2].grad}


# --------------------------------------------------------------------- exact
def exact(case, seed):
    c = dict(DEFAULTS, **case)
    sim = _simulation(c)
    prob, x = sim["prob"], _member(sim, seed)
    size = prob.nelem * prob.nlev
    if c["kind"] in ("step", "coupled"):
        # the member's first pass
        m = _Model(prob, "cuda")
        v, T, ps = x
        qdp = torch.as_tensor(_tracers(sim, seed)[:, 0, :c["qsize"]], device="cuda")
        f = make_forcing(prob, seed) if c["kind"] == "coupled" else None
        f = f and {k: torch.as_tensor(a, device="cuda") for k, a in f.items()}
        for _ in range(c["calls"]):
            v, T, ps, qdp, Q, omega = m.interval(v, T, ps, qdp, f)
        if c["kind"] == "step":
            return {"v": v, "T": T, "ps": ps, "qdp": qdp.transpose(0, 1).contiguous()}
        return {"v": v, "T": T, "ps": ps, "dp3d": None, "qdp": qdp, "Q": Q, "omega_p": omega}
    if size * c["calls"] * c["qsplit"] * max(c["rsplit"], 1) > 16 * 16 * 6 * 72 * 2:
        return None
    m = _Model(prob, "cuda")
    if c["kind"] == "adjoint":
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        lam = [torch.randn(a.shape, generator=g, dtype=torch.float64, device="cuda") for a in x]
        lam = m.pull_back(x, lam)
        return {"v": lam[0], "T": lam[1], "ps": lam[2]}
    states = [x]
    for _ in range(c["calls"]):
        states.append(tuple(a.detach() for a in m.dry(*states[-1])))
    end = states[-1]
    # the mismatch is quadratic: its gradients in closed form
    (vt, Tt, pt), w = synthetic_target(prob, seed), region_weight(prob)
    g, cp, rgas, t_ref, p_ref = 9.80616, 1005.0, 287.04, 300.0, 1.0e5
    wk = w[:, None] * m.reference_thickness() / g
    we = w * (rgas * t_ref / p_ref / g)
    d = end[0] - vt, end[1] - Tt, end[2] - pt
    lam = [wk[:, :, None] * d[0], wk * (cp / t_ref) * d[1], we * d[2]]
    loss = 0.5 * sum((a * b).sum() for a, b in zip(lam, d))
    for s in reversed(states[:-1]):
        lam = m.pull_back(s, lam)
    return {"loss": loss, "v": end[0], "T": end[1], "ps": end[2], "gv": lam[0], "gT": lam[1], "gps": lam[2]}


class _Model:
    """The step in plain torch: fields (nelem, nlev, 4, 4), winds with the
    component third, tracers (nelem, qsize, nlev, 4, 4)."""

    RD, RV, CP, RRE = 287.04, 461.5, 1005.0, 1.0 / 6.376e6

    def __init__(self, prob, device):
        def t(a):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=device)

        self.p, self.dt, self.L, self.device = prob.params, prob.dt, prob.nlev, device
        m, vc = prob.metric, prob.vcoord
        self.D, self.Di, self.mi = (t(m[k]).unsqueeze(3).unbind(1) for k in ("D", "Dinv", "metinv"))
        self.D, self.Di, self.mi = ([r.unbind(1) for r in a] for a in (self.D, self.Di, self.mi))
        self.md, self.sph, self.rsph, self.mp, self.f = (t(m[k])[:, None] for k in (
            "metdet", "spheremp", "rspheremp", "mp", "fcor"))
        self.phis, self.dvv = t(prob.state["phis"])[:, None], t(prob.dvv)
        self.ps0, self.top = vc.ps0, float(vc.hyai[0] * vc.ps0)
        self.da, self.db = (t(np.diff(a)).view(-1, 1, 1) for a in (vc.hyai, vc.hybi))
        self.hybi = t(vc.hybi).view(-1, 1, 1)
        key = np.round(prob.mesh.pos * 1e9).astype(np.int64).reshape(-1, 3)
        _, node = np.unique(key, axis=0, return_inverse=True)
        self.node, self.nodes = torch.as_tensor(node.reshape(-1), device=device), int(node.max()) + 1

    def reference_thickness(self):
        return (self.da + self.db) * self.ps0

    # operators of an element: derivatives along the two reference directions
    def dx(self, s, mat=None):
        return s @ (self.dvv if mat is None else mat).T

    def dy(self, s, mat=None):
        return self.dx(s.transpose(-1, -2), mat).transpose(-1, -2)

    def grad(self, s):
        a, b, Di = self.dx(s) * self.RRE, self.dy(s) * self.RRE, self.Di
        return Di[0][0] * a + Di[0][1] * b, Di[1][0] * a + Di[1][1] * b

    def div(self, a, b):
        Di = self.Di
        x = self.md * (Di[0][0] * a + Di[1][0] * b)
        y = self.md * (Di[0][1] * a + Di[1][1] * b)
        return (self.dx(x) + self.dy(y)) * (self.RRE / self.md)

    def vorticity(self, u, v):
        D = self.D
        return (self.dx(D[1][0] * u + D[1][1] * v) - self.dy(D[0][0] * u + D[0][1] * v)) * (self.RRE / self.md)

    def laplace(self, s):
        a, b = self.grad(s)
        Di = self.Di
        x = self.sph * (Di[0][0] * a + Di[1][0] * b)
        y = self.sph * (Di[0][1] * a + Di[1][1] * b)
        return -self.RRE * (self.dx(x, self.dvv.T) + self.dy(y, self.dvv.T))

    def vector_laplace(self, u, v, ratio):
        D, mi = self.D, self.mi
        s = self.mp * self.div(u, v) * ratio
        a, b = self.dx(s, self.dvv.T), self.dy(s, self.dvv.T)
        x = -self.md * (mi[0][0] * a + mi[0][1] * b)
        y = -self.md * (mi[1][0] * a + mi[1][1] * b)
        s = self.mp * self.vorticity(u, v)
        x, y = x + self.dy(s, self.dvv.T), y - self.dx(s, self.dvv.T)
        k = 2.0 * self.sph * self.RRE ** 2
        return k * u + (D[0][0] * x + D[1][0] * y) * self.RRE, k * v + (D[0][1] * x + D[1][1] * y) * self.RRE

    def assemble(self, s):
        n = s.shape[1]
        flat = s.permute(0, 2, 3, 1).reshape(-1, n)
        whole = torch.zeros(self.nodes, n, dtype=s.dtype, device=s.device).index_add(0, self.node, flat)
        return whole[self.node].view(-1, 4, 4, n).permute(0, 3, 1, 2)

    def project(self, s):
        return self.rsph * self.assemble(s)

    def thickness(self, ps):
        return self.da * self.ps0 + self.db * ps[:, None]

    # dynamics
    def stage(self, base, at, h, qv, flux, weight):
        (v0, T0, d0), (vel, T, dp) = base, at
        u, v = vel.unbind(2)
        div = self.div(u * dp, v * dp)
        above = torch.cumsum(div, 1) - div
        p = self.top + torch.cumsum(dp, 1) - 0.5 * dp
        Tv = T if qv is None else T * (1.0 + (self.RV / self.RD - 1.0) * qv / dp)
        r = self.RD * Tv * (0.5 * dp / p)
        phi = self.phis + 2.0 * torch.flip(torch.cumsum(torch.flip(r, [1]), 1), [1]) - r
        px, py = self.grad(p)
        omega = (u * px + v * py - above - 0.5 * div) / p
        up, down, etas = 0.0, 0.0, 0.0

        def vertical(s):
            return 0.0

        if self.p.rsplit == 0:
            total = above[:, -1:] + div[:, -1:]
            eta = self.hybi[:-1] * total - above
            zero = torch.zeros_like(eta[:, :1])
            down = torch.cat([zero, eta[:, 1:]], 1)
            up = torch.cat([eta[:, 1:], zero], 1)
            etas = up - down

            def vertical(s):
                step = 0.5 * (s[:, 1:] - s[:, :-1])
                z = torch.zeros_like(s[:, :1])
                return (up * torch.cat([step, z], 1) + down * torch.cat([z, step], 1)) / dp

        tx, ty = self.grad(T)
        Tn = T0 + h * (self.RD / self.CP * Tv * omega - u * tx - v * ty - vertical(T))
        ex, ey = self.grad(0.5 * (u * u + v * v) + phi)
        k, z = self.RD * Tv / p, self.vorticity(u, v) + self.f
        un = v0[:, :, 0] + h * (v * z - ex - k * px - vertical(u))
        vn = v0[:, :, 1] + h * (-u * z - ey - k * py - vertical(v))
        dn = d0 - h * (div + etas)
        if flux is not None and weight:
            flux["v"] = flux["v"] + weight * vel * dp[:, :, None]
            flux["omega"] = flux["omega"] + weight * omega
        un, vn, Tn, dn = (self.project(self.sph * a) for a in (un, vn, Tn, dn))
        return torch.stack([un, vn], 2), Tn, dn

    def smooth(self, x, flux, weight):
        p, dt = self.p, self.dt / self.p.hypervis_subcycle
        ratio = p.nu_div / p.nu
        vel, T, dp = x
        u, v = vel.unbind(2)
        a, b, c, d = (self.project(s) for s in (*self.vector_laplace(u, v, ratio), self.laplace(T), self.laplace(dp)))
        a, b = self.vector_laplace(a, b, ratio)
        c, d = self.laplace(c), self.laplace(d)
        if flux is not None:
            flux["dp"] = flux["dp"] + weight * dp / p.hypervis_subcycle
            flux["bih"] = flux["bih"] + weight * d / p.hypervis_subcycle
        sponge = torch.zeros(self.L, 1, 1, dtype=T.dtype, device=T.device)
        sponge[:3, 0, 0] = p.nu_top * torch.tensor([4.0, 2.0, 1.0], dtype=T.dtype, device=T.device)[:self.L]
        su, sv = self.vector_laplace(u, v, 1.0)
        a, b = sponge * su - p.nu * a, sponge * sv - p.nu * b
        c, d = sponge * self.laplace(T) - p.nu_s * c, sponge * self.laplace(dp) - p.nu_p * d
        a, b, c = (dt * self.project(s) for s in (a, b, c))
        un, vn = u + a, v + b
        return torch.stack([un, vn], 2), T + c - (a * un + b * vn) / self.CP, self.project(self.sph * dp + dt * d)

    def dynamics(self, x, qv=None, flux=None, share=1.0):
        h = self.dt
        a = self.stage(x, x, h / 5, qv, flux, share / 4)
        b = self.stage(x, a, h / 5, qv, flux, 0)
        b = self.stage(x, b, h / 3, qv, flux, 0)
        b = self.stage(x, b, 2 * h / 3, qv, flux, 0)
        w = tuple((5.0 * s - t) / 4.0 for s, t in zip(a, x))
        x = self.stage(w, b, 3 * h / 4, qv, flux, 3 * share / 4)
        for _ in range(self.p.hypervis_subcycle):
            x = self.smooth(x, flux, share)
        return x

    # tracers
    def bounds(self, q):
        return q.amin((-1, -2)), q.amax((-1, -2))

    def neighbours(self, lo, hi):
        """bounds over each element and those that share a point with it"""
        n = lo.shape[0]
        el = torch.arange(n, device=lo.device).repeat_interleave(16)

        def spread(s, how):
            s = s.reshape(n, -1)
            i = self.node[:, None].expand(-1, s.shape[1])
            at = torch.empty(self.nodes, s.shape[1], dtype=s.dtype, device=s.device)
            at = at.scatter_reduce(0, i, s[el], how, include_self=False)
            at = at[self.node].view(n, 16, -1)
            return (at.amin(1) if how == "amin" else at.amax(1)).view(lo.shape)

        return spread(lo, "amin"), spread(hi, "amax")

    def limit(self, x, c, lo, hi):
        s1 = c.sum((-1, -2), keepdim=True)
        s0 = (x * c).sum((-1, -2), keepdim=True)
        lo, hi = lo[..., None, None].clamp(min=0), hi[..., None, None]
        lo = torch.where(s0 < lo * s1, s0 / s1, lo)
        hi = torch.where(s0 > hi * s1, s0 / s1, hi)
        if self.p.limiter_option == 9:
            y = torch.minimum(torch.maximum(x, lo), hi)
            add = ((x - y) * c).sum((-1, -2), keepdim=True)
            room = torch.where(add > 0, hi - y, y - lo)
            fac = (c * room).sum((-1, -2), keepdim=True)
            x = torch.where((add != 0) & (fac > 0), y + add / fac * room, y)
        else:
            going = torch.ones_like(s0, dtype=torch.bool)
            for _ in range(15):
                y = torch.minimum(torch.maximum(x, lo), hi)
                add = ((x - y) * c).sum((-1, -2), keepdim=True)
                x = torch.where(going, y, x)
                going = going & (add.abs() > 5e-14 * s0.abs())
                if not going.any():
                    break
                free = torch.where(add > 0, x < hi, x > lo)
                fac = torch.where(free, c.expand_as(x), 0.0).sum((-1, -2), keepdim=True)
                x = torch.where(going & free, x + add / fac, x)
        return x, lo[..., 0, 0], hi[..., 0, 0]

    def tracers(self, qdp, dp0, flux):
        """three stages of the transport over one tracer step"""
        p, dt = self.p, 0.5 * self.dt * self.p.qsplit
        u, v = flux["v"].unbind(2)
        div = self.div(u, v)
        proj = self.project(self.sph * div)
        start = qdp
        for stage in range(3):
            dp = dp0 - stage * dt * (div if stage == 0 else proj)
            q = qdp / dp[:, None]
            if stage == 1:
                a, b = self.bounds(q)
                lo, hi = torch.minimum(lo, a), torch.maximum(hi, b)
            else:
                lo, hi = self.neighbours(*self.bounds(q))
            left, add = dp - dt * div, 0.0
            if stage == 2:
                left = left - 3.0 * dt * p.nu_q * flux["bih"] / self.sph
                ref = self.reference_thickness()
            nxt = torch.empty_like(qdp)
            for i in range(qdp.shape[1]):
                if stage == 2:
                    s = self.laplace(self.project(self.laplace(q[:, i] * flux["dp"] / ref)))
                    add = -3.0 * dt * p.nu_q * ref * s / self.sph
                x = qdp[:, i] - dt * self.div(u / dp * qdp[:, i], v / dp * qdp[:, i]) + add
                y, lo[:, i], hi[:, i] = self.limit(x / left, self.sph * left, lo[:, i], hi[:, i])
                nxt[:, i] = self.project(self.sph * left * y)
            qdp = nxt
        return (start + 2.0 * qdp) / 3.0

    # remap
    def remap(self, fields, src, tgt):
        """column integrals of the fields' parabolas: fields, src and tgt
        (nelem, nlev, 4, 4), each field a mass per layer"""
        L, alg = self.L, self.p.remap_alg

        def ghosts(s):
            return torch.cat([s[:, 1:2], s[:, :1], s, s[:, -1:], s[:, -2:-1]], 1)

        d = ghosts(src)
        zero = torch.zeros_like(src[:, :1])
        edge = torch.cat([zero, torch.cumsum(src, 1)], 1)
        aim = torch.cumsum(tgt, 1).detach() if not tgt.requires_grad else torch.cumsum(tgt, 1)
        aim = torch.cat([aim[:, :-1], edge[:, -1:]], 1)
        with torch.no_grad():
            cell = torch.searchsorted(edge.movedim(1, -1).contiguous(), aim.movedim(1, -1).contiguous(), right=True)
            cell = (cell - 1).clamp(0, L - 1).movedim(-1, 1)
        width = src.gather(1, cell)
        z = (aim - 0.5 * (edge.gather(1, cell) + edge.gather(1, cell + 1))) / width
        m, c, n = d[:, :-2], d[:, 1:-1], d[:, 2:]
        s0, s1, s2 = c / (m + c + n), (2 * m + c) / (c + n), (c + 2 * n) / (m + c)
        m, c, n, o = d[:, :-3], d[:, 1:-2], d[:, 2:-1], d[:, 3:]
        e1, e2 = c / (c + n), 1.0 / (m + c + n + o)
        e3 = 2.0 * c * n / (c + n) * ((m + c) / (2 * c + n) - (o + n) / (2 * n + c))
        e4, e5 = c * (m + c) / (2 * c + n), n * (n + o) / (c + 2 * n)
        out = []
        for s in fields:
            a = ghosts(s / src)
            up, dn = a[:, 2:] - a[:, 1:-1], a[:, 1:-1] - a[:, :-2]
            g = s0 * (s1 * up + s2 * dn)
            small = torch.minimum(g.abs(), 2.0 * torch.minimum(up.abs(), dn.abs()))
            g = torch.where(up * dn > 0, small * torch.sign(g), 0.0)
            step = a[:, 2:-1] - a[:, 1:-2]
            face = a[:, 1:-2] + e1 * step + e2 * (e3 * step - e4 * g[:, 1:] + e5 * g[:, :-1])
            a, l, r = a[:, 2:-2], face[:, :-1], face[:, 1:]
            flat = (r - a) * (a - l) <= 0
            l, r = torch.where(flat, a, l), torch.where(flat, a, r)
            l = torch.where((r - l) * (a - 0.5 * (l + r)) > (r - l) ** 2 / 6, 3 * a - 2 * r, l)
            r = torch.where((r - l) * (a - 0.5 * (l + r)) < -(r - l) ** 2 / 6, 3 * a - 2 * l, r)
            c0, c1, c2 = 1.5 * a - 0.25 * (l + r), r - l, 3.0 * (l + r) - 6.0 * a
            if alg == 2:
                ends = torch.zeros(L, 1, 1, dtype=torch.bool, device=s.device)
                ends[:2] = ends[-2:] = True
                c0, c1, c2 = torch.where(ends, a, c0), torch.where(ends, 0.0, c1), torch.where(ends, 0.0, c2)
            c0, c1, c2 = (k.gather(1, cell) for k in (c0, c1, c2))
            part = c0 * (z + 0.5) + 0.5 * c1 * (z * z - 0.25) + c2 * (z ** 3 + 0.125) / 3
            mass = torch.cat([zero, torch.cumsum(s, 1)], 1).gather(1, cell) + part * width
            out.append(torch.cat([mass[:, :1], mass[:, 1:] - mass[:, :-1]], 1))
        return out

    def settle(self, x):
        """end of a remap interval: states on the levels of the new ps"""
        vel, T, dp = x
        ps = self.top + dp.sum(1)
        if self.p.rsplit == 0:
            return vel, T, ps
        tgt = self.thickness(ps)
        u, v, T = (s / tgt for s in self.remap([vel[:, :, 0] * dp, vel[:, :, 1] * dp, T * dp], dp, tgt))
        return torch.stack([u, v], 2), T, ps

    def dry(self, v, T, ps):
        x = (v, T, self.thickness(ps))
        for _ in range(self.p.qsplit * max(self.p.rsplit, 1)):
            x = self.dynamics(x)
        return self.settle(x)

    def pull_back(self, x, lam):
        x = [a.detach().requires_grad_() for a in x]
        return torch.autograd.grad(self.dry(*x), x, lam)

    def interval(self, v, T, ps, qdp, forcing=None):
        """one remap interval with tracers (Lagrangian levels): v, T, ps, Qdp, Q, omega"""
        p = self.p
        span = self.dt * p.qsplit * p.rsplit
        if forcing:
            T, v = T + span * forcing["FT"], v + span * forcing["FM"]
            qdp = qdp + torch.maximum(span * forcing["FQ"][:, :qdp.shape[1]], -qdp)
        x = (v, T, self.thickness(ps))
        for _ in range(p.rsplit):
            z = torch.zeros_like(T)
            flux, dp0 = {"v": torch.zeros_like(v), "omega": z, "dp": z, "bih": z}, x[2]
            for _ in range(p.qsplit):
                x = self.dynamics(x, qdp[:, 0] if p.moisture else None, flux, 1.0 / p.qsplit)
            qdp = self.tracers(qdp, dp0, flux)
        v, T, ps = self.settle(x)
        tgt = self.thickness(ps)
        qdp = torch.stack(self.remap(qdp.unbind(1), x[2], tgt), 1)
        return v, T, ps, qdp, qdp / tgt[:, None], self.project(self.sph * flux["omega"])
