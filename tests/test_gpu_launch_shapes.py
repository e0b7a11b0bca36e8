"""Launch shapes chosen by size.  The deposit kernels sum each cell's particles
in bin order whatever the rows and planes a block takes, so the built-in shape
of every grid size must give the state that a fixed long march gives, bit for
bit: the smallest grid, sides where the rule stops at one wave, at single
planes and at one row, and unequal sides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 16, 16), (8, 32, 16), (64, 32, 64), (16, 8, 512)])
def test_built_in_deposit_shape_equals_a_fixed_one(gpu_available, shape):
    import tpx
    from tpx import ic
    nz, ny, nx = shape
    npart = nx * ny * nz // 2 + 3
    case = ic.make_case(nx, npart, nu=0.05, seed=5, St=1.0, phi=0.3, heat=True, eps_range=(0.5, 1.0), drag_limit=True,
                        shape=shape)
    out = []
    for fixed in (False, True):
        s = tpx.Solver(case.params, np_capacity=npart)
        if fixed:
            s.set_tiles(heat=(1, 8), velocity=(1, 8))
        s.load_case(case)
        s.step(2)
        out.append((s.get("RU"), s.get("Rho"), s.particles(), s.rhs_t()))
        s.close()
    (ru, rho, p, h), (ru1, rho1, p1, h1) = out
    assert np.isfinite(ru).all()
    assert np.array_equal(ru, ru1) and np.array_equal(rho, rho1) and np.array_equal(h, h1)
    for k in p:
        assert np.array_equal(p[k], p1[k]), k
