"""The calls of this framework whose time is measured, over the range its users run.

A user holds a solver (tpx.Solver) with the state uploaded, advances it a
stretch of RK4 steps and fetches what is stored or analysed: the gas momentum,
density and pressure and every particle (the reference's slow dump).  Beside
that, an ensemble of small boxes advanced together (tpx.Batch), the adjoint of
a stretch of steps (record, then every gradient), and the Poisson solve with a
caller's face coefficient on device arrays.

Kinds of case
  step      `steps` whole RK4 steps of one box, then the state
  ensemble  `steps` steps of `boxes` boxes by batched kernels, then their momentum
  adjoint   a recorded stretch of `steps` steps (checkpoints every `every`) and
            every gradient of the variance of the final particle concentration
  solve     one Poisson solve with the caller's coefficient, device to device

A pass of the first three continues the run where the last pass left it, as a
driver loop does.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "triplyperiodic-modified_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import tpx  # noqa: E402
from tpx.params import PI, Params  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
PRE = (0.5, 0.5, 1.0, 1.0 / 6.0)
POST = (1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0)
PART_Q = ("x", "y", "z", "u", "v", "w", "T")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _step(name, nx, ny, nz, np_, steps, st=1.0, spread=False, phi=0.2, heat=False, twc=True, cooling=False,
          gravity=0.0, flow=0.0, rho_var=0.0, passive=False):
    """One box: Stokes number `st` (`spread`: per particle, log-uniform in
    [0.1, 10]), mass loading `phi`, the heat exchange with per-particle
    absorption (`heat`), the gas held at its energy (`cooling`), gravity (in
    units of u'^2 over the height) and a mean flow along x, an initial density of relative spread `rho_var`, a
    passive scalar and a passive vector (`passive`)."""
    return dict(name=name, kind="step", nx=nx, ny=ny, nz=nz, particles=np_, steps=steps, st=st, spread=spread, phi=phi,
                heat=heat, twc=twc, cooling=cooling, gravity=gravity, flow=flow, rho_var=rho_var, passive=passive)


def listed():
    return [
        # the Poisson solve by itself for a caller on the GPU: a small grid,
        # where launches and the wait on the stopping test count, and the
        # largest grid that the entry point takes
        dict(name="solve_32", kind="solve", nx=32, ny=32, nz=32, spread=0.5),
        dict(name="solve_128", kind="solve", nx=128, ny=128, nz=128, spread=0.5),
        # the smallest configuration: 32^3, 16,384 two-way coupled particles
        _step("plain_32", 32, 32, 32, 16384, 40),
        # one box of an ensemble's size run by itself, an odd particle count
        _step("box_64", 64, 64, 64, 44721, 30, st=0.7, phi=0.3),
        # the middle configuration: 128^3, 1e6 particles of spread Stokes numbers
        _step("plain_128", 128, 128, 128, 1_000_000, 24, spread=True, phi=0.5),
        # unequal sides with every term of the step: heat exchange with the
        # energy balanced, gravity, mean flow, variable density
        _step("terms_128x32x64", 128, 32, 64, 100_003, 20, st=1.5, phi=0.4, heat=True, cooling=True, gravity=0.5,
              flow=0.25, rho_var=0.1),
        # a long box (the grid's longest axis, 512), one-way coupled tracers in
        # gas of variable density
        _step("long_512x64x128", 512, 64, 128, 250_007, 12, st=0.3, twc=False, rho_var=0.2),
        # single-phase gas carrying a passive scalar and a passive vector
        _step("passive_128", 128, 128, 128, 0, 12, passive=True),
        # the headline configuration: 256^3, 1.6e7 heated particles
        _step("heat_256", 256, 256, 256, 16_000_000, 32, phi=1.0, heat=True),
        # the ensemble: 64 boxes of 64^3, uneven particle counts
        dict(name="ensemble_64x64", kind="ensemble", n=64, boxes=64, steps=24),
        # the adjoint with the heat exchange, the gas replayed segment by segment
        dict(name="adjoint_128", kind="adjoint", n=128, particles=200_000, steps=20, every=10, heat=True,
             tape="segments"),
        # the adjoint of a small box without heat, the gas tape kept in memory
        dict(name="adjoint_64", kind="adjoint", n=64, particles=25_001, steps=10, every=5, heat=False, tape="auto"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of these ranges: sides 16 to 512 (powers of two, as the
    solver takes), particle counts of any parity from none to several a cell,
    each option on or off, and a cost below the headline configuration's."""
    kind = rng.choice(["step"] * 7 + ["solve"] * 2 + ["ensemble", "adjoint", "adjoint"])
    if kind == "ensemble":
        return dict(kind="ensemble", n=rng.choice([32, 64]), boxes=rng.randint(3, 48), steps=rng.randint(6, 20))
    if kind == "adjoint":
        n = rng.choice([32, 64, 64, 128])
        steps = rng.randint(4, 14)
        return dict(kind="adjoint", n=n, particles=_logint(rng, 2e3, 0.1 * n ** 3 + 4e3) | 1, steps=steps,
                    every=rng.randint(2, steps), heat=rng.random() < 0.5,
                    tape=rng.choice(["auto", "segments", "recompute"]))
    top = 1 << 21 if kind == "solve" else 1 << 23
    while True:
        nx, ny, nz = (1 << rng.randint(4, 9) for _ in range(3))
        if 8192 <= nx * ny * nz <= top and max(nx, ny, nz) <= 16 * min(nx, ny, nz):
            break
    if kind == "solve":
        return dict(kind="solve", nx=nx, ny=ny, nz=nz, spread=round(rng.uniform(0.1, 1.0), 3))
    cells = nx * ny * nz
    gas = rng.random() < 0.2
    heat = not gas and rng.random() < 0.5
    c = _step("", nx, ny, nz, 0 if gas else _logint(rng, 0.02 * cells + 100, 1.2 * cells), rng.randint(5, 24),
              st=round(math.exp(rng.uniform(math.log(0.3), math.log(5.0))), 3), spread=rng.random() < 0.3,
              phi=round(rng.uniform(0.1, 0.8), 3), heat=heat, twc=rng.random() < 0.7,
              cooling=heat and rng.random() < 0.5, gravity=round(rng.uniform(0.1, 1.0), 3) if rng.random() < 0.4 else 0.0,
              flow=0.25 if rng.random() < 0.3 else 0.0,
              rho_var=round(rng.uniform(0.05, 0.2), 3) if rng.random() < 0.5 else 0.0, passive=rng.random() < 0.15)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs (made on the GPU from the seed; numpy arrays for the solver's uploads)
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _wave(shape, L):
    nz, ny, nx = shape
    k = [torch.fft.fftfreq(n, d=1.0 / n, dtype=F64, device=DEV) * (2 * math.pi / l)
         for n, l in ((nz, L[2]), (ny, L[1]))]
    kx = torch.arange(nx // 2 + 1, dtype=F64, device=DEV) * (2 * math.pi / L[0])
    return kx[None, None, :], k[1][None, :, None], k[0][:, None, None]


def _filtered(shape, L, k0, g):
    """A real random field of spectrum k^4 exp(-2 (k/k0)^2), zero mean."""
    kx, ky, kz = _wave(shape, L)
    k = torch.sqrt(kx * kx + ky * ky + kz * kz)
    amp = k * torch.exp(-(k / k0) ** 2)
    return torch.fft.rfftn(torch.randn(shape, generator=g, dtype=F64, device=DEV)) * amp


def _velocity(shape, L, k0, g):
    """Random solenoidal face velocity (discretely divergence free on the
    staggered grid), u' = 1: the spectral initial condition of the benchmark
    configurations."""
    nz, ny, nx = shape
    d = (L[0] / nx, L[1] / ny, L[2] / nz)
    K = _wave(shape, L)
    uh = [_filtered(shape, L, k0, g) for _ in range(3)]
    bwd = [(1 - torch.exp(-1j * K[c] * d[c])) / d[c] for c in range(3)]  # grad_C2F
    lap = sum((2 / d[c] ** 2) * (1 - torch.cos(K[c] * d[c])) for c in range(3)).clone()
    lap[0, 0, 0] = 1.0
    phi = sum(-bwd[c].conj() * uh[c] for c in range(3)) / -lap  # div_F2C = -conj(grad_C2F)
    u = torch.stack([torch.fft.irfftn(uh[c] - bwd[c] * phi, s=shape) for c in range(3)])
    return u / torch.sqrt((u * u).sum(0).mean() / 3)


def _roll(f, axis, n):  # axis 0, 1, 2 = x, y, z; n = +1 takes the upper neighbour
    return torch.roll(f, -n, dims=2 - axis)


def _dissipation(u, nu, d):
    sq = 0.0
    for a in range(3):
        sq += float((((_roll(u[a], a, 1) - u[a]) / d[a]) ** 2).mean())
        for b in range(a + 1, 3):
            s = 0.5 * ((u[a] - _roll(u[a], b, -1)) / d[b] + (u[b] - _roll(u[b], a, -1)) / d[a])
            sq += 2 * float((s * s).mean())
    return 2 * nu * sq


def _gather_u(u, pos, L):
    nz, ny, nx = u.shape[1:]
    N = (nx, ny, nz)
    s = [pos[c] * (N[c] / L[c]) for c in range(3)]
    i0 = [(s[c].long()) % N[c] for c in range(3)]
    fr = [s[c] - s[c].floor() for c in range(3)]
    flat = u.reshape(3, -1)
    at = lambda i: (i[2] * ny + i[1]) * nx + i[0]  # noqa: E731
    out = []
    for c in range(3):
        i1 = list(i0)
        i1[c] = (i0[c] + 1) % N[c]
        out.append(fr[c] * flat[c][at(i1)] + (1 - fr[c]) * flat[c][at(i0)])
    return out


def _box(nx, ny, nz, npart, seed, st=1.0, spread=False, phi=0.2, heat=False, twc=True, cooling=False, gravity=0.0,
         flow=0.0, rho_var=0.0, passive=False, nu=None):
    """Parameters and initial state of one box by the benchmark recipe: dt from
    CFL 0.3, viscosity scaled to the grid, Lundgren forcing at the initial
    dissipation, particles uniform with the gas velocity."""
    g = _gen(seed)
    shape, nmin = (nz, ny, nx), min(nx, ny, nz)
    h = 2 * PI / nmin
    L = (h * nx, h * ny, h * nz)
    nu = 0.64 / nmin if nu is None else nu
    u = _velocity(shape, L, min(4.0, nmin / 8.0), g)
    d = (h, h, h)
    eps0 = _dissipation(u, nu, d)
    tau_eta = math.sqrt(nu / eps0)
    u[0] += flow
    p = Params(Nx_tot=nx, Ny_tot=ny, Nz_tot=nz, Lx=L[0], Ly=L[1], Lz=L[2], bs=2)
    p.dt = 0.3 / (max(float(u[c].max()) for c in range(3)) / h)
    p.Mu0, p.Rho0, p.T0, p.Cp, p.Cv = nu, 1.0, 1.0, 3.5, 2.5
    p.Cvp = p.Cv
    p.k = p.Mu0 * p.Cp / 0.7
    # forced where the box bounds the largest eddies; decaying in a long box
    p.A1 = p.A2 = eps0 / 3 if nx == ny == nz else 0.0
    p.TWC, p.cooling = int(twc), int(cooling)
    p.Iteration1 = p.Iteration2 = 50
    p.epsilon = 1e-10
    p.U0 = flow
    if gravity:
        p.gz1 = p.gz2 = -gravity / L[2]
        p.ParticleGravity = 1
    vol = L[0] * L[1] * L[2]
    s = dict(params=p)
    tau = eps = None
    parts = None
    if npart:
        mp = phi * vol / npart
        p.Dp = mp / (3 * PI * p.Mu0 * st * tau_eta)
        p.Rhop = 6 * mp / (PI * p.Dp ** 3)
        p.np0 = (npart + 0.5) / vol
        smin = st
        if spread:
            ln = torch.rand(npart, generator=g, dtype=F64, device=DEV) * math.log(100.0)
            tau = 0.1 * torch.exp(ln) * st * tau_eta
            smin = 0.1 * st
        if twc:  # the coupled drag of a cell's gas and several particles stays resolved
            p.dt = min(p.dt, smin * tau_eta / (1.0 + 4.0 * mp / h ** 3))
        else:
            p.dt = min(p.dt, smin * tau_eta)
        if heat:
            p.Nu = 2.0
            p.I01 = p.I02 = 4 * (0.5 * p.Nu * PI * p.Dp * p.k) / (0.75 * PI * p.Dp ** 2)
            eps = 0.5 + 0.5 * torch.rand(npart, generator=g, dtype=F64, device=DEV)
            # as the drag: the rate at which a particle warms its cell's gas
            rate = p.Nu * PI * p.Dp * p.k / (p.Cp * h ** 3)
            p.dt = min(p.dt, 0.25 / rate)
            # the lamp warms a cell that holds a particle by at most some
            # hundredths a step (a tenth of that where the gas is held at its
            # energy, so that the parts without particles do not cool away)
            per_cell = npart / (nx * ny * nz)
            step = 0.5 * p.dt * rate * p.Cp / p.Cv * per_cell
            p.I01 = p.I02 = p.I01 * min(1.0, (0.001 if cooling else 0.01) * min(1.0, per_cell) / step)
        pos = [torch.rand(npart, generator=g, dtype=F64, device=DEV) * L[c] for c in range(3)]
        parts = pos + _gather_u(u, pos, L) + [torch.ones(npart, dtype=F64, device=DEV)]
    rho = torch.ones(shape, dtype=F64, device=DEV)
    if rho_var:
        f = torch.fft.irfftn(_filtered(shape, L, min(3.0, nmin / 8.0), g), s=shape)
        rho = rho + rho_var * f / (3 * f.std())
    face = lambda c: 0.5 * (rho + _roll(rho, c, -1))  # noqa: E731
    s.update(RU=torch.stack([u[c] * face(c) for c in range(3)]), Rho=rho, parts=parts, tau=tau, eps=eps)
    if passive:
        p.solve_for_scalar = p.solve_for_vector = 1
        p.s1t, p.s2t, p.D_M, p.eta, p.Rho_forV = 0.0, 0.0, nu, nu, 1.0
        s["PS"] = torch.fft.irfftn(_filtered(shape, L, min(3.0, nmin / 8.0), g), s=shape)
        s["PS"] /= s["PS"].std()
        s["RV"] = _velocity(shape, L, min(3.0, nmin / 8.0), g)
    return s


def _solver(s):
    """A solver with the state uploaded and initialised."""
    n = 0 if s["parts"] is None else s["parts"][0].numel()
    sim = tpx.Solver(s["params"], np_capacity=n)
    sim.set("RU", s["RU"].cpu().numpy())
    sim.set("Rho", s["Rho"].cpu().numpy())
    sim.set("P", np.zeros(tuple(s["Rho"].shape)))
    if n:
        host = [q.cpu().numpy() for q in s["parts"]]
        sim.set_particles(*host, np.arange(n, dtype=np.int32), tau=None if s["tau"] is None else s["tau"].cpu().numpy(),
                          eps=None if s["eps"] is None else s["eps"].cpu().numpy())
    if "PS" in s:
        sim.set("Passive_Scalar", s["PS"].cpu().numpy())
        sim.set("RV", s["RV"].cpu().numpy())
        sim.set("Q", np.zeros(tuple(s["Rho"].shape)))
    sim.set_restart_numbers(s["params"].P0, 0.0, 0)
    sim.initialize()
    return sim


def _step_box(case, seed):
    a = {k: case[k] for k in ("nx", "ny", "nz", "st", "spread", "phi", "heat", "twc", "cooling", "gravity", "flow",
                              "rho_var", "passive")}
    return _box(npart=case["particles"], seed=seed, **a)


def _ensemble_boxes(case, seed):
    """Boxes of one size with viscosity, Stokes number and particle count of
    their own: counts log-uniform over a factor of 20, as in the 64 x 64^3
    configuration."""
    r = np.random.default_rng(seed + 4242)
    n, out = case["n"], []
    for b in range(case["boxes"]):
        nu = r.uniform(0.01, 0.03) * 64 / n
        st = math.exp(r.uniform(math.log(0.1), math.log(10.0)))
        npart = int(math.exp(r.uniform(math.log(1e4), math.log(2e5))) * n ** 3 / 64 ** 3)
        out.append(_box(n, n, n, npart, seed * 1000 + b, st=st, phi=0.3, nu=nu))
    return out


def _adjoint_box(case, seed):
    n = case["n"]
    return _box(n, n, n, case["particles"], seed, st=2.0, phi=0.5, heat=case["heat"])


def _solve_inputs(case, seed):
    """A face coefficient in [1, 1 + spread], a right-hand side that has a
    solution (the operator on a random field) and an initial guess."""
    g = _gen(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    h = 2 * PI / case["nx"]
    P = torch.randn(shape, generator=g, dtype=F64, device=DEV)
    C = [1 + case["spread"] * torch.rand(shape, generator=g, dtype=F64, device=DEV) for _ in range(3)]
    rhs = _div([C[c] * _grad(P, c, h) for c in range(3)], (h, h, h))
    P0 = 0.1 * torch.randn(shape, generator=g, dtype=F64, device=DEV)
    return C, rhs, P0, h


def prepare(case, seed):
    if case["kind"] == "step":
        return dict(kind="step", sim=_solver(_step_box(case, seed)), steps=case["steps"],
                    particles=case["particles"] > 0, passive=case["passive"])
    if case["kind"] == "ensemble":
        sims = [_solver(s) for s in _ensemble_boxes(case, seed)]
        return dict(kind="ensemble", sims=sims, batch=tpx.Batch(sims), steps=case["steps"])
    if case["kind"] == "adjoint":
        sim = _solver(_adjoint_box(case, seed))
        sim.adjoint_set_gas_tape(case["tape"])
        return dict(kind="adjoint", sim=sim, steps=case["steps"], every=case["every"])
    C, rhs, P0, h = _solve_inputs(case, seed)
    p = Params(Nx_tot=case["nx"], Ny_tot=case["ny"], Nz_tot=case["nz"], Lx=h * case["nx"], Ly=h * case["ny"],
               Lz=h * case["nz"], bs=2, dt=1e-2, Iteration1=50, Iteration2=50, epsilon=1e-10, TWC=0)
    sim = tpx.Solver(p, np_capacity=1)
    fn = sim.L.tpx_poisson_solve_device
    fn.argtypes = [ctypes.c_void_p] * 6 + [ctypes.POINTER(ctypes.c_int)]
    return dict(kind="solve", sim=sim, fn=fn, C=C, rhs=rhs, P0=P0, P=torch.empty_like(P0), its=ctypes.c_int(0))


def run(state):
    kind = state["kind"]
    if kind == "step":
        sim = state["sim"]
        sim.step(state["steps"])
        out = dict(RU=sim.get("RU"), Rho=sim.get("Rho"), P=sim.get("P"), P0=sim.scalars()["P0"])
        if state["particles"]:
            out["particles"] = sim.particles()
        if state["passive"]:
            out.update(PS=sim.get("Passive_Scalar"), RV=sim.get("RV"), Q=sim.get("Q"))
        return out
    if kind == "ensemble":
        state["batch"].step(state["steps"])
        return [sim.get("RU") for sim in state["sims"]]
    if kind == "adjoint":
        sim = state["sim"]
        J = sim.adjoint_record(state["steps"], state["every"])
        out = dict(J=J, **sim.adjoint_gradient_full())
        # the solves converge from any start: their result does not depend on
        # the initial P, whose gradient is round-off around zero
        del out["P"]
        return out
    # the solve runs on the solver's own stream: the guess has to be in place
    state["P"].copy_(state["P0"])
    torch.cuda.current_stream().synchronize()
    ptr = [t.data_ptr() for t in state["C"] + [state["P"], state["rhs"]]]
    rc = state["fn"](state["sim"].h, *ptr, ctypes.byref(state["its"]))
    if rc != 0:
        raise RuntimeError(state["sim"].L.tpx_last_error(state["sim"].h).decode())
    return dict(P=state["P"], iterations=state["its"].value)


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------
def _step_work(cells, npart, heat, twc, passive):
    """One RK4 step: per substep the momentum and density update (reads the
    stage, base and running momentum and density, writes the next ones; 20
    values a cell), the Poisson right-hand side (5), at least one Poisson
    iteration (P, density and right-hand side read, P written: 4) and the
    projection (13); per particle the stage, base and running state (21 read,
    14 written) and, with coupling or heat, the deposited fields."""
    cell = 20 + 5 + 4 + 13 + (6 if npart and twc else 0) + (2 if npart and heat else 0) + (36 if passive else 0)
    part = 35 + (3 if twc else 0) + (2 if heat else 0)
    fl = cells * (220 + 60 * math.log2(max(2, cells))) + npart * (120 + (90 if heat else 0))
    return 4 * 8.0 * (cell * cells + part * npart), 4.0 * fl


def work(case):
    if case["kind"] == "solve":
        n = case["nx"] * case["ny"] * case["nz"]
        # coefficient, right-hand side and guess read, the pressure written;
        # a variable coefficient takes some ten iterations of two transforms
        return dict(bytes=8.0 * 6 * n, flops=10.0 * n * (40 + 5 * math.log2(n)))
    if case["kind"] == "ensemble":
        n = case["n"] ** 3
        b, f = _step_work(n, n * 0.25, False, True, False)
        m = case["boxes"] * case["steps"]
        return dict(bytes=m * b + case["boxes"] * 24.0 * n, flops=m * f)
    if case["kind"] == "adjoint":
        n = case["n"] ** 3
        b, f = _step_work(n, case["particles"], case["heat"], True, False)
        # forward and reverse: each at least a step's own work
        return dict(bytes=2 * case["steps"] * b + 8.0 * (5 * n + 8 * case["particles"]), flops=2 * case["steps"] * f)
    n = case["nx"] * case["ny"] * case["nz"]
    b, f = _step_work(n, case["particles"], case["heat"], case["twc"], case["passive"])
    out = 8.0 * (n * (10 if case["passive"] else 5) + 7.5 * case["particles"])
    return dict(bytes=case["steps"] * b + out, flops=case["steps"] * f)


# ---------------------------------------------------------------------------
# the same results in plain torch, 64 bits (functional, so that autograd
# gives the adjoint's gradients)
# ---------------------------------------------------------------------------
def _grad(f, c, h):
    return (f - _roll(f, c, -1)) / h


def _div(F, d):
    return sum((_roll(F[c], c, 1) - F[c]) / d[c] for c in range(3))


def _lap(f, d):
    return sum((_roll(f, c, 1) - 2 * f + _roll(f, c, -1)) / d[c] ** 2 for c in range(3))


def _face(f, c):
    return 0.5 * (f + _roll(f, c, -1))


class _Exact:
    """The solver's step on torch tensors (nz, ny, nx), vectors as lists."""

    def __init__(self, p, tau=None, eps=None):
        self.p, self.tau, self.eps = p, tau, eps
        self.N = (p.Nx_tot, p.Ny_tot, p.Nz_tot)
        self.L = (p.Lx, p.Ly, p.Lz)
        self.d = tuple(l / n for l, n in zip(self.L, self.N))
        self.vcell = self.d[0] * self.d[1] * self.d[2]
        K = _wave((p.Nz_tot, p.Ny_tot, p.Nx_tot), self.L)
        lam = sum((2 / self.d[c] ** 2) * (1 - torch.cos(K[c] * self.d[c])) for c in range(3)).clone()
        lam[0, 0, 0] = 1.0  # the zero mode is passed through
        self.lam = lam
        self.heat = p.Nu * p.Dp * p.k != 0

    # ---- Poisson ----
    def solve(self, C, P, rhs):
        p, d = self.p, self.d
        cc = -3.0 / sum(0.5 * (C[c] + _roll(C[c], c, 1)) for c in range(3))
        its, err = 0, 100.0
        while its < p.Iteration1 and err > p.epsilon:
            r = (_div([_grad(P, c, d[c]) * C[c] for c in range(3)], d) - rhs) * cc
            dp = -torch.fft.irfftn(torch.fft.rfftn(r) / self.lam, s=r.shape)
            P = P + dp
            err = float(dp.detach().abs().max())
            its += 1
        return P, its

    # ---- particles ----
    def cell(self, i):
        return (torch.remainder(i[2], self.N[2]) * self.N[1] + torch.remainder(i[1], self.N[1])) * self.N[0] + \
            torch.remainder(i[0], self.N[0])

    def floor(self, x):
        s = [x[c] / self.d[c] for c in range(3)]
        i = [v.detach().long() for v in s]
        return i, [v - j for v, j in zip(s, i)]

    def cic(self, x):
        """The eight corners (flat cell, weight) of each particle."""
        s = [x[c] / self.d[c] for c in range(3)]
        i = [torch.floor(v.detach() + 0.5).long() for v in s]
        f = [v - j + 0.5 for v, j in zip(s, i)]
        for a in (0, 1):
            for b in (0, 1):
                for e in (0, 1):
                    w = (f[0] if a else 1 - f[0]) * (f[1] if b else 1 - f[1]) * (f[2] if e else 1 - f[2])
                    yield self.cell([i[0] - 1 + a, i[1] - 1 + b, i[2] - 1 + e]), w

    def deposit(self, x, v):
        out = torch.zeros(self.N[0] * self.N[1] * self.N[2], dtype=F64, device=x[0].device)
        for at, w in self.cic(x):
            out = out.index_add(0, at, w if v is None else w * v)
        return out.reshape(self.N[2], self.N[1], self.N[0])

    def exchange(self, x, T, rho, P0):
        p = self.p
        Tg = ((P0 / p.R) / rho).reshape(-1)
        tg = sum(w * Tg[at] for at, w in self.cic(x))
        rt = (tg - T) * (p.Nu * PI * p.Dp * p.k)
        return rt, self.deposit(x, rt)

    def init(self, RU, rho, P, P0, parts=None, PS=None, RV=None):
        s = dict(RU=list(RU), RUi=list(RU), rho=rho, rhoi=rho, P=P, P0=P0, P0i=P0, Q=torch.zeros_like(rho))
        if parts is not None:
            order = torch.sort(self.cell(self.floor([q.detach() for q in parts[:3]])[0]), stable=True)[1]
            s["order"] = order
            s["q"] = [v[order] for v in parts]
            s["tau"] = None if self.tau is None else self.tau[order]
            s["eps"] = None if self.eps is None else self.eps[order]
            s["rt"] = torch.zeros_like(s["q"][6])
            if self.heat:
                s["rt"], s["Q"] = self.exchange(s["q"][:3], s["q"][6], rho, P0)
            s["qi"] = list(s["q"])
        if PS is not None:
            s.update(PS=PS, PSi=PS, RV=list(RV), RVi=list(RV), Qv=torch.zeros_like(rho))
        return s

    def substep(self, s, rk):
        """One RK4 substep: s holds base, int (…i) and running np1 (…1) values."""
        p, d = self.p, self.d
        a, b = p.dt * POST[rk], p.dt * PRE[rk]
        last = rk == 3
        o = dict(s)
        F = [_face(s["rhoi"], c) for c in range(3)]
        U = [s["RUi"][c] / F[c] for c in range(3)]
        div_ru = _div(s["RUi"], d)
        o["rho1"] = s["rho1"] - a * div_ru
        rho = o["rho1"] if last else s["rho"] - b * div_ru
        dP0 = 0.0 if p.cooling else -p.R / p.Cv * s["Q"].mean() / self.vcell
        o["P01"] = s["P01"] + a * dP0
        P0 = o["P01"] if last else s["P0"] + b * dP0
        S = None
        if "q" in s:
            xi, vi = s["qi"][:3], s["qi"][3:6]
            i, f = self.floor(xi)
            lo, hi, gas = self.cell(i), [], []
            for c in range(3):
                j = list(i)
                j[c] = j[c] + 1
                hi.append(self.cell(j))
                u = U[c].reshape(-1)
                gas.append(f[c] * u[hi[c]] + (1 - f[c]) * u[lo])
            itp = 1 / p.Tp if s["tau"] is None else 1 / s["tau"]
            drag = [(gas[c] - vi[c]) * itp for c in range(3)]
            g = [p.ParticleGravity * v for v in (p.gx1, p.gy1, p.gz1)]
            e = p.epsilonp if s["eps"] is None else s["eps"]
            rate = list(vi) + [drag[c] + g[c] for c in range(3)] + \
                [(s["rt"] + 0.25 * e * PI * p.Dp ** 2 * p.I01) / (p.mp * p.Cvp)]
            q1 = [s["q1"][k] + a * rate[k] for k in range(7)]
            qn = list(q1) if last else [s["q"][k] + b * rate[k] for k in range(7)]
            base = list(s["q"])
            if p.TWC:
                n = U[0].numel()
                S = []
                for c in range(3):
                    v = torch.zeros(n, dtype=F64, device=DEV).index_add(0, hi[c], f[c] * drag[c])
                    S.append(v.index_add(0, lo, (1 - f[c]) * drag[c]).reshape(U[0].shape))
            for c in range(3):
                x = qn[c].detach()
                sh = (x < 0).to(F64) * self.L[c] - (x > self.L[c]).to(F64) * self.L[c]
                qn[c], q1[c], base[c] = qn[c] + sh, q1[c] + sh, base[c] + sh
            o["q"], o["q1"], o["qi"] = base, q1, qn
            if self.heat:
                o["rt"], o["Q"] = self.exchange(qn[:3], qn[6], rho, P0)
        if "PS" in s:
            self.passive(s, o, U, F, a, b, last, rk)
        div_u = _div(U, d)
        RUn = []
        o["RU1"] = list(s["RU1"])
        for c in range(3):
            r = p.Mu0 / 3 * _grad(div_u, c, d[c]) + p.Mu0 * _lap(U[c], d) + p.A1 * s["RUi"][c]
            r = r + (p.gx1, p.gy1, p.gz1)[c] * (F[c] - p.Rho0)
            if S is not None:
                r = r - p.mp / self.vcell * S[c]
            r = r - _div([_face(U[c], e) * _face(s["RUi"][e], c) for e in range(3)], d)
            o["RU1"][c] = s["RU1"][c] + a * r
            RUn.append(o["RU1"][c] if last else s["RU"][c] + b * r)
        Q = o["Q"] - o["Q"].mean() if p.cooling else o["Q"]
        div = p.k / p.Cp * _lap(1 / rho, d) - p.R / (p.Cp * P0 * self.vcell) * Q
        F = [_face(rho, c) for c in range(3)]
        rhs = (_div([RUn[c] / F[c] for c in range(3)], d) - div) / b
        o["P"], _ = self.solve([1 / F[c] for c in range(3)], s["P"], rhs - rhs.mean())
        for c in range(3):
            gp = _grad(o["P"], c, d[c])
            o["RU1"][c] = o["RU1"][c] - a * gp
            RUn[c] = o["RU1"][c] if last else RUn[c] - b * gp
        o["rhoi"], o["RUi"], o["P0i"] = rho, RUn, P0
        return o

    def passive(self, s, o, U, F, a, b, last, rk):
        """The passive scalar (source cos x less its mean) and the passive
        vector (source cos x on the y component less its mean)."""
        p, d = self.p, self.d
        X = d[0] / 2 + torch.arange(self.N[0], dtype=F64, device=DEV) * d[0]
        src = (torch.cos(X) - torch.cos(X).mean())[None, None, :]
        r = p.D_M * _lap(s["PSi"], d) - _div([U[c] * _face(s["PSi"], c) for c in range(3)], d) + src
        o["PS1"] = s["PS1"] + a * r
        o["PSi"] = o["PS1"] if last else s["PS"] + b * r
        V = [v / p.Rho_forV for v in s["RVi"]]
        dv = _div(V, d)
        new = []
        o["RV1"] = list(s["RV1"])
        for c in range(3):
            r = p.eta / 3 * _grad(dv, c, d[c]) + p.eta * _lap(V[c], d)
            r = r - _div([_face(s["RVi"][c], e) * _face(U[e], c) for e in range(3)], d)
            if c == 1:
                r = r + src
            o["RV1"][c] = s["RV1"][c] + a * r
            new.append(o["RV1"][c] if last else s["RV"][c] + b * r)
        rhs = _div([v / p.Rho_forV for v in new], d) / b
        one = torch.full_like(rhs, 1 / p.Rho_forV)
        o["Qv"], _ = self.solve([one] * 3, s["Qv"], rhs - rhs.mean())
        for c in range(3):
            gp = _grad(o["Qv"], c, d[c])
            o["RV1"][c] = o["RV1"][c] - a * gp
            new[c] = o["RV1"][c] if last else new[c] - b * gp
        o["RVi"] = new

    def step(self, s, substep=None):
        p = self.p
        s = dict(s, RU1=list(s["RU"]), rho1=s["rho"], P01=s["P0"])
        if "q" in s:
            s["q1"] = list(s["q"])
        if "PS" in s:
            s["PS1"], s["RV1"] = s["PS"], list(s["RV"])
        for rk in range(4):
            s = (substep or self.substep)(s, rk)
        mean = (p.U0 * p.Rho0, p.V0 * p.Rho0, p.W0 * p.Rho0)
        s["RU"] = [s["RU1"][c] - s["RU1"][c].mean() + mean[c] for c in range(3)]
        s["rho"], s["P0"] = s["rho1"], s["P01"]
        if "PS" in s:
            s["PS"], s["RV"] = s["PS1"], list(s["RV1"])
        if "q" in s:
            s["q"] = list(s["q1"])
            if p.TWC or self.heat:  # the particles are kept in cell order
                at = torch.sort(self.cell(self.floor([q.detach() for q in s["q"][:3]])[0]), stable=True)[1]
                for k in ("tau", "eps", "rt", "order"):
                    s[k] = None if s[k] is None else s[k][at]
                s["q"] = [v[at] for v in s["q"]]
                s["qi"] = list(s["q"])
        return s


def _exact_run(box, steps):
    p = box["params"]
    m = _Exact(p, box["tau"], box["eps"])
    P0 = torch.tensor(p.P0, dtype=F64, device=DEV)
    s = m.init([box["RU"][c] for c in range(3)], box["Rho"], torch.zeros_like(box["Rho"]), P0, box["parts"],
               box.get("PS"), box.get("RV"))
    for _ in range(steps):
        s = m.step(s)
    return s


def _exact_adjoint(box, steps):
    """Every gradient by autograd through the steps, a substep at a time."""
    from torch.utils.checkpoint import checkpoint
    p = box["params"]
    leaf = lambda t: t.detach().clone().requires_grad_(True)  # noqa: E731
    npart = box["parts"][0].numel()
    RU, rho = [leaf(box["RU"][c]) for c in range(3)], leaf(box["Rho"])
    P, P0 = torch.zeros_like(box["Rho"]), leaf(torch.tensor(p.P0, dtype=F64, device=DEV))
    q, A = [leaf(v) for v in box["parts"]], leaf(torch.tensor(p.A1, dtype=F64, device=DEV))
    tau = leaf(torch.full((npart,), p.Tp, dtype=F64, device=DEV))
    eps = None if box["eps"] is None else leaf(box["eps"])

    class Pars:  # the parameters with the forcing coefficient as a tensor
        A1 = A

        def __getattr__(self, k):
            return getattr(p, k)

    m = _Exact(Pars(), tau, eps)
    s = m.init(RU, rho, P, P0, q)

    def flat(s):
        keys, vals = [], []
        for k in sorted(s):
            for j, v in enumerate(s[k] if isinstance(s[k], list) else [s[k]]):
                keys.append((k, isinstance(s[k], list)))
                vals.append(v)
        return keys, vals

    def unflat(keys, vals):
        s = {}
        for (k, many), v in zip(keys, vals):
            if many:
                s.setdefault(k, []).append(v)
            else:
                s[k] = v
        return s

    def sub(s, rk):
        keys, vals = flat(s)
        out_keys = []

        def f(*v):
            k, o = flat(m.substep(unflat(keys, v), rk))
            out_keys[:] = k
            return tuple(o)

        return unflat(out_keys, checkpoint(f, *vals, use_reentrant=False))

    for _ in range(steps):
        s = m.step(s, sub)
    C = m.deposit(s["q"][:3], None)
    J = (C * C).mean() - C.mean() ** 2
    J.backward()
    at, z = s["order"], torch.zeros(npart, dtype=F64, device=DEV)
    g = lambda t: z if t.grad is None else t.grad  # noqa: E731
    out = dict(J=float(J.detach()), tau=g(tau)[at], state=torch.stack([g(v)[at] for v in q[:6]]), A=float(A.grad),
               RU=torch.stack([v.grad for v in RU]), Rho=rho.grad)
    if m.heat:
        out.update(T=g(q[6])[at], eps=eps.grad[at], P0=float(P0.grad))
    return out


def exact(case, seed):
    if case["kind"] == "solve":
        C, rhs, P, h = _solve_inputs(case, seed)
        n = (case["nx"], case["ny"], case["nz"])
        p = Params(Nx_tot=n[0], Ny_tot=n[1], Nz_tot=n[2], Lx=h * n[0], Ly=h * n[1], Lz=h * n[2], Iteration1=50,
                   epsilon=1e-10)
        P, its = _Exact(p).solve(C, P, rhs)
        return dict(P=P, iterations=its)
    if case["kind"] == "ensemble":
        if case["boxes"] * case["steps"] > 1600:
            return None
        return [torch.stack(_exact_run(b, case["steps"])["RU"]) for b in _ensemble_boxes(case, seed)]
    if case["kind"] == "adjoint":
        if case["steps"] * case["n"] ** 3 > 20 * 128 ** 3:
            return None
        return _exact_adjoint(_adjoint_box(case, seed), case["steps"])
    # some 0.1 microseconds a particle and step for the deposits
    if case["steps"] * (case["nx"] * case["ny"] * case["nz"] + 4 * case["particles"]) > 1.5e8:
        return None
    s = _exact_run(_step_box(case, seed), case["steps"])
    out = dict(RU=torch.stack(s["RU"]), Rho=s["rho"], P=s["P"], P0=float(s["P0"]))
    if case["particles"]:
        out["particles"] = dict(zip(PART_Q, s["q"]), flag=s["order"].to(torch.int32))
    if case["passive"]:
        out.update(PS=s["PS"], RV=torch.stack(s["RV"]), Q=s["Qv"])
    return out
