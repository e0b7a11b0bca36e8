"""The momentum kernel's march length: single planes where two would leave fewer
than 256 blocks.  Its stencil keeps the reference's operand order, so every
march length must give the oracle's bits: the smallest grid, the last shapes
that take single planes and the first that take two."""
import numpy as np
import pytest

from test_gpu_parity import _noncubic_case, oracle_from_case, solver_from_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 16, 64), (64, 32, 32), (32, 64, 32), (64, 32, 64)])
def test_momentum_bits(gpu_available, shape):
    case = _noncubic_case(shape, seed=53)
    o, s = oracle_from_case(case), solver_from_case(case)
    o.set_rk4_count(0)
    for m in ("update_rho", "update_p0", "update_particle", "update_ru_wop"):
        getattr(o, m)()
        getattr(s, m)(0)
    for q in ("Rho_new", "Rho_np1", "RU_new", "RU_np1"):
        assert np.array_equal(s.get(q), o.get(q)), q
