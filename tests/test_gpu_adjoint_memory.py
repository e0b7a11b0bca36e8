"""Device memory of adjoint recordings of different lengths on one solver: a
short recording after a long one holds what it would hold by itself, beside at
most 1 GiB kept from the other (here none: the long one holds more), in every
tape form; and the short one's gradients are those of a solver of its own."""
import ctypes

import numpy as np
import pytest

from helpers import small_case, solver_from_case

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def _free():
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so.7")  # the runtime libtpx is linked to
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("tape,steps", [("keep", 12), ("recompute", 24), ("segments", 48)])
def test_short_recording_after_a_long_one(gpu_available, tape, steps):
    case = small_case(n=64, npart=20000, seed=3)
    a, b = solver_from_case(case), solver_from_case(case)
    for s in (a, b):
        s.adjoint_set_gas_tape(tape)
    b.step(steps)
    held, out = [], []
    for s, lengths in ((b, (1,)), (a, (steps, 1))):
        before = _free()
        for n in lengths:
            s.adjoint_record(n, n)
            g = s.adjoint_gradient_full()
            held.append(before - _free())
        out.append(g)
        s.adjoint_release()
    a.close()
    b.close()
    alone, long_one, after = held
    print(tape, f"alone {alone / GIB:.2f} GiB, {steps} steps {long_one / GIB:.2f}, 1 step after them {after / GIB:.2f}")
    assert long_one > GIB + alone
    assert after <= alone + (32 << 20)  # the runtime's granularity
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
