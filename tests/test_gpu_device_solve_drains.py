"""tpx_poisson_solve_device hands the caller's arrays back idle.  The second
solve of each pair starts at the first one's result and stops after fewer
iterations than were queued for it: the leftover ones read the arrays, and when
the call returns they have gone from the solver's stream.  Shapes of the
three-pass form (full-length and packed rows) and, with an axis of 8, of the
five-pass form."""
import ctypes

import numpy as np
import pytest

from test_oracle_poisson_coef import manufactured

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (16, 32, 64), (128, 128, 128), (16, 8, 64)])
def test_nothing_is_in_flight_after_the_call(gpu_available, shape):
    from test_zz_no_alloc import DeviceArrays
    from tpx import Solver
    p, _, C, RHS = manufactured(shape, seed=sum(shape), spread=0.5)
    p.epsilon, p.Iteration1, p.Iteration2 = 1e-10, 50, 50
    s = Solver(p, np_capacity=1)
    L, its = s.L, ctypes.c_int(0)
    L.tpx_poisson_solve_device.argtypes = [ctypes.c_void_p] * 6 + [ctypes.POINTER(ctypes.c_int)]
    dev = DeviceArrays([C[0], C[1], C[2], np.zeros(shape), RHS])
    query, stream, counts = dev.hip.hipStreamQuery, ctypes.c_void_p(s.stream()), []
    query.argtypes = [ctypes.c_void_p]
    try:
        for _ in range(2):
            rc = L.tpx_poisson_solve_device(s.h, *dev.ptrs, ctypes.byref(its))
            left = query(stream)
            assert rc == 0
            counts.append(its.value)
    finally:
        dev.free()
    s.close()
    assert counts[0] > counts[1] >= 1, counts
    assert left == 0  # hipSuccess: the stream is empty
