"""Axes of 512 in the three-pass Poisson iteration (lengths 16..512, y and z not
both 512): the spectral step against numpy-style transforms in long double, whole
gas steps against the oracle and the five-pass form, the adjoint's replays
against its stored iterates, and coefficient solves whose second pass has the
largest runs, or whose arrays the packed rows must not be given.

Bounds, u = 2^-53.  A transform of N points errs by at most 8 u (log2 N + 2) of
its input's 2-norm (4 sqrt(2) + 2 roundings a level, two levels more for the
packed real rows); division by lambda amplifies what the forward transform left
by 1 / lambda_min; lambda itself is 2/d^2 (1 - cos), off by up to 4 u times the
sum of 2/d^2 in the library and in the reference.  A converged solve is off by
the residual's rounding, 12 roundings of the sum T of its terms' magnitudes,
divided by the operator: for the largest values of both, at most 1.25 /
lambda_min (a square wave along the longest axis), and the mean mode, which is
passed through, gathers one such rounding an iteration.  Two solutions differ by
twice that; over the substeps of a step the error of RU, dt grad P, comes back
through the next right-hand side, at most doubling each time (1 + 2 + 4 + 8)."""
import ctypes

import numpy as np
import pytest
import scipy.fft

from helpers import oracle_from_case, solver_from_case
from test_gpu_coef_three_pass import _case as coef_case
from test_gpu_parity import _noncubic_case

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _spacing(p):
    return np.array([p.Lx / p.Nx_tot, p.Ly / p.Ny_tot, p.Lz / p.Nz_tot])


def _lambda(p):
    """The modified wavenumbers of poisson.cpp:433-449 on the full spectrum."""
    d, out = _spacing(p), 0.0
    for a, n in enumerate((p.Nx_tot, p.Ny_tot, p.Nz_tot)):
        k = np.fft.fftfreq(n, 1.0 / n)
        lam = 2.0 / d[a] ** 2 * (1.0 - np.cos(2 * np.pi / n * k))
        out = out + lam.reshape([-1 if b == 2 - a else 1 for b in range(3)])
    return out


@pytest.mark.parametrize("shape", [(16, 16, 512), (16, 64, 512), (16, 256, 512), (16, 512, 16), (32, 512, 16),
                                   (64, 512, 32), (128, 512, 16), (256, 512, 16), (512, 16, 16), (512, 64, 16),
                                   (512, 128, 16), (512, 16, 512)])
def test_spectral_step(gpu_available, shape):
    case = _noncubic_case((16, 16, 16), seed=1)
    p = case.params
    p.Nz_tot, p.Ny_tot, p.Nx_tot = shape
    p.Lx, p.Ly, p.Lz = 2 * np.pi, 2 * np.pi * shape[1] / shape[2], 2 * np.pi * shape[0] / shape[2]
    from tpx import Solver
    s = Solver(p, np_capacity=1)
    x = np.random.default_rng(5).standard_normal(shape)
    got, _ = s.adjoint_check(0, x, x)
    s.close()
    lam = _lambda(p)
    lam[0, 0, 0] = 1.0  # the mean mode is passed through
    X = scipy.fft.fftn(x.astype(np.longdouble), norm="ortho")
    Y = X / lam
    ref = -scipy.fft.ifftn(Y, norm="ortho").real
    tr = 8 * U * (np.log2(x.size) + 2)
    norm = lambda v: float(np.sqrt(np.sum(np.abs(v) ** 2)))  # noqa: E731
    bound = tr * norm(x) / min(1.0, float(lam.min())) + (tr + 4 * U) * norm(ref)
    bound += 4 * U * float(np.sum(2.0 / _spacing(p) ** 2)) * norm(Y / lam)
    err = norm(got - ref)
    print(shape, f"error {err:.2e} of {norm(ref):.2e}, bound {bound:.2e}")
    assert err <= bound <= 1e-6 * norm(ref)


def _solve_bound(p, P, rho_range, rhs_max, iterations, coef_max):
    d, T = _spacing(p), 0.0
    for a in range(3):
        g = np.abs(P - np.roll(P, 1, axis=2 - a)) / d[a]
        T = T + (g + np.roll(g, -1, axis=2 - a)) / d[a]
    T = (float(T.max()) * coef_max + rhs_max) * rho_range
    lam = _lambda(p)
    lam[0, 0, 0] = np.inf
    return 12 * U * T * (1.25 / float(lam.min()) + iterations)


@pytest.mark.parametrize("shape", [(16, 16, 512), (16, 64, 512), (16, 512, 16), (32, 512, 64), (512, 16, 16)])
def test_gas_step(gpu_available, monkeypatch, shape):
    case = _noncubic_case(shape, seed=sum(shape))
    p = case.params
    s3, o = solver_from_case(case), oracle_from_case(case)
    monkeypatch.setenv("TPX_FFT_PASSES", "5")
    s5 = solver_from_case(case)
    for q in (s3, s5, o):
        q.step(1)
    its = s3.scalars()["num_iteration"]
    assert its == s5.scalars()["num_iteration"] == o.scalars()["num_iteration"] < 50
    lo, hi = float(case.Rho.min()), float(case.Rho.max())
    tol = 2 * 15 * _solve_bound(p, o.get("P"), hi, float(np.abs(s5.get("RHS_Pois")).max()), its, 1.0 / lo)
    h = float(_spacing(p).min())
    tol_ru = p.dt * 2 / h * tol + 64 * U * float(np.abs(o.get("RU")).max())
    tol_rho = 4 * p.dt * 6 / h * tol_ru + 64 * U * hi
    for name, t in (("P", tol), ("RU", tol_ru), ("Rho", tol_rho)):
        ref = o.get(name)
        e3, e5 = np.max(np.abs(s3.get(name) - ref)), np.max(np.abs(s3.get(name) - s5.get(name)))
        m = float(np.max(np.abs(ref)))
        print(shape, name, f"oracle {e3 / m:.2e} five passes {e5 / m:.2e} bound {t / m:.2e}")
        assert max(e3, e5) <= t <= 1e-6 * m
    s3.close()
    s5.close()


@pytest.mark.parametrize("shape", [(128, 512, 16), (256, 512, 16)])
def test_coefficient_solve_with_the_largest_runs(gpu_available, monkeypatch, shape):
    p, C, RHS, P0 = coef_case(shape)
    from tpx import Solver
    out = []
    for passes in ("3", "5"):
        monkeypatch.setenv("TPX_FFT_PASSES", passes)
        s = Solver(p, np_capacity=1)
        out.append(s.poisson_solve(C, P0, RHS))
        s.close()
    (P3, i3), (P5, i5) = out
    tol = 2 * _solve_bound(p, P5, 1.0, float(np.abs(RHS).max()), i5, float(C.max()))
    e, m = float(np.max(np.abs(P3 - P5))), float(np.max(np.abs(P5)))
    print(shape, f"difference {e / m:.2e} bound {tol / m:.2e} iterations", i3)
    assert i3 == i5 > 2 and e <= tol <= 1e-6 * m


@pytest.mark.parametrize("off", [1, 2, 3])
def test_device_arrays_of_any_alignment(gpu_available, monkeypatch, off):
    """An x length of 512 has only packed rows in the three-pass form: arrays
    that are not 16-byte aligned (odd offsets) take the five passes."""
    from test_zz_no_alloc import DeviceArrays
    from tpx import Solver
    shape = (16, 16, 512)
    p, C, RHS, P0 = coef_case(shape)
    s = Solver(p, np_capacity=1)
    ref, its = s.poisson_solve(C, P0, RHS)
    n = int(np.prod(shape))
    padded = np.zeros((5, n + 4))
    for q, a in enumerate((C[0], C[1], C[2], P0, RHS)):
        padded[q, off:off + n] = np.asarray(a).reshape(-1)
    dev = DeviceArrays(list(padded))
    L, got = s.L, ctypes.c_int(0)
    L.tpx_poisson_solve_device.argtypes = [ctypes.c_void_p] * 6 + [ctypes.POINTER(ctypes.c_int)]
    try:
        rc = L.tpx_poisson_solve_device(s.h, *[q.value + 8 * off for q in dev.ptrs], ctypes.byref(got))
        whole = dev.get(3) if rc == 0 else None
    finally:
        dev.free()
    s.close()
    tol = 2 * _solve_bound(p, ref, 1.0, float(np.abs(RHS).max()), its, float(C.max()))
    assert rc == 0 and got.value == its
    e = float(np.max(np.abs(whole[off:off + n].reshape(shape) - ref)))
    print(off, f"difference {e:.2e} bound {tol:.2e}")
    assert e <= tol and not whole[:off].any() and not whole[off + n:].any()


@pytest.mark.parametrize("shape", [(16, 16, 512), (16, 512, 16), (512, 16, 16)])
def test_adjoint_replays(gpu_available, shape):
    """A recording that keeps the Poisson iterates, one that recomputes each
    step (every iteration out of place) and one that replays segments give the
    same gradients bit for bit."""
    case = _noncubic_case(shape, seed=7 + sum(shape))
    p, rng, npart = case.params, np.random.default_rng(11), 600
    vol = p.Lx * p.Ly * p.Lz
    mp = 0.2 * vol / np.prod(shape)  # a fifth of a cell's gas
    p.TWC = 1
    p.dt = min(p.dt, 0.05 * float(_spacing(p).min()) ** 2 / p.Mu0)  # the explicit diffusion stays stable over the steps
    p.Dp = mp / (3 * np.pi * p.Mu0 * 0.05)
    p.Rhop = 6 * mp / (np.pi * p.Dp ** 3)
    p.np0 = (npart + 0.5) / vol
    case.RU *= 0.2
    case.particles = {q: rng.uniform(0, l, npart) for q, l in zip("xyz", (p.Lx, p.Ly, p.Lz))}
    case.particles.update({q: 0.3 * rng.standard_normal(npart) for q in "uvw"})
    case.particles.update(T=np.full(npart, p.T0), flag=np.arange(npart, dtype=np.int32))
    out = []
    for tape in ("keep", "recompute", "segments"):
        s = solver_from_case(case)
        s.adjoint_set_gas_tape(tape)
        J = s.adjoint_record(3, 2)
        out.append(dict(J=np.array(J), **s.adjoint_gradient_full()))
        s.close()
    for other in out[1:]:
        for k, v in out[0].items():
            assert np.all(np.isfinite(v)) and np.any(v != 0.0), k
            assert np.array_equal(v, other[k]), k
