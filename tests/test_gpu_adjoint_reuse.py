"""Recordings that take over the memory of earlier ones: a second recording on
the same solver (same size, shorter, longer, another tape) gives, bit for bit,
the gradients that a solver of its own gives for the same state, and leaves the
deposits where the run ended."""
import numpy as np
import pytest

from helpers import small_case, solver_from_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heat", [False, True])
@pytest.mark.parametrize("tapes", [("segments", "segments"), ("keep", "recompute"), ("recompute", "keep")])
def test_second_recording_equals_a_first_one(gpu_available, heat, tapes):
    case = small_case(n=16, npart=700, heat=heat, variable_rho=True, eps_range=(0.5, 1.0) if heat else None, seed=3)
    a, b = solver_from_case(case), solver_from_case(case)
    steps = (4, 3, 5)
    a.adjoint_set_gas_tape(tapes[0])
    for n in steps[:2]:
        a.adjoint_record(n, 2)
        a.adjoint_gradient_full()
    b.step(steps[0] + steps[1])
    got = []
    for s in (a, b):
        s.adjoint_set_gas_tape(tapes[1])
        J = s.adjoint_record(steps[2], 2)
        g = s.adjoint_gradient_full()
        got.append((J, g, s.get("RHS_RU"), s.get("RHS_Part_Temp"), s.get("RU")))
        s.adjoint_release()
    (J, g, S, Q, RU), (J1, g1, S1, Q1, RU1) = got
    assert J == J1 and np.array_equal(S, S1) and np.array_equal(Q, Q1) and np.array_equal(RU, RU1)
    for k in g:
        assert np.array_equal(g[k], g1[k]), k
    a.close()
    b.close()
