"""The coefficient Poisson solve's three-pass iteration (its residual formed in
the first pass) against the residual kernel and the five passes
(TPX_FFT_PASSES=5): the same operations up to the order of the transforms'
sums, so the same iterations and results within 1e-12.  Sides that take the
packed rows (64, 128, 256), the full-length rows of 16 lanes and fewer, the
smallest and unequal ones; and device arrays that are not 16-byte aligned,
which the packed rows must not be given."""
import ctypes

import numpy as np
import pytest

from test_oracle_poisson_coef import manufactured

pytestmark = pytest.mark.gpu


def _solver(p, monkeypatch, passes):
    from tpx import Solver
    monkeypatch.setenv("TPX_FFT_PASSES", passes)
    return Solver(p, np_capacity=1)


def _case(shape):
    p, _, C, RHS = manufactured(shape, seed=sum(shape), spread=0.5)
    p.epsilon, p.Iteration1, p.Iteration2 = 1e-10, 50, 50
    return p, C, RHS, 0.1 * np.random.default_rng(7).standard_normal(shape)


@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 16, 32), (16, 64, 64), (64, 16, 128), (16, 32, 256), (256, 32, 16),
                                   (16, 8, 64), (512, 16, 16), (16, 16, 512), (16, 512, 32), (512, 128, 16),
                                   (16, 512, 512), (32, 256, 512)])
def test_three_pass_coefficient_solve_equals_five_pass(gpu_available, monkeypatch, shape):
    p, C, RHS, P0 = _case(shape)
    out = []
    for passes in ("3", "5"):
        s = _solver(p, monkeypatch, passes)
        out.append(s.poisson_solve(C, P0, RHS))
        s.close()
    (P3, i3), (P5, i5) = out
    assert i3 == i5 > 2
    assert np.max(np.abs(P3 - P5)) <= 1e-12 * np.max(np.abs(P5))


@pytest.mark.parametrize("off", [0, 1, 3])
def test_unaligned_device_arrays(gpu_available, monkeypatch, off):
    from test_zz_no_alloc import DeviceArrays
    shape = (16, 32, 64)
    p, C, RHS, P0 = _case(shape)
    s = _solver(p, monkeypatch, "3")
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
        P = dev.get(3)[off:off + n].reshape(shape) if rc == 0 else None
    finally:
        dev.free()
    s.close()
    assert rc == 0 and got.value == its
    assert np.max(np.abs(P - ref)) <= 1e-12 * np.max(np.abs(ref))
