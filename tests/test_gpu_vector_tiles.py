"""Update_RV_WOQ's tiles against the oracle: the smallest sides, where a tile
spans the whole box and wraps onto itself, sides below, at and above the tile's
32 x 8, and marches of 2 to 16 planes.  The kernel keeps the reference's
operands and order, so its update agrees with the oracle's to the last bits:
1e-14 of the largest value (64 roundings of 1.1e-16 a value, most of which
coincide)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s2t", [0.0, 1.0])
@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 16, 8), (16, 8, 32), (8, 32, 16), (64, 16, 32), (32, 32, 64), (16, 8, 256)])
def test_update_rv_woq_against_the_oracle(gpu_available, shape, s2t):
    import tpx
    from oracle.oracle import Oracle
    from tpx import ic
    nz, ny, nx = shape
    case = ic.make_case(nx, 0, nu=0.05, seed=2, shape=shape)
    p = case.params
    p.solve_for_vector, p.s2t, p.eta, p.Rho_forV = 1, s2t, 0.03, 1.3
    rng = np.random.default_rng(sum(shape))
    rho = 1.0 + 0.2 * rng.random(shape)
    rv = rng.standard_normal((3,) + shape)
    o, s = Oracle(p.struct_fields()), tpx.Solver(p)
    for m in (o, s):
        m.set("RU", case.RU)
        m.set("Rho", rho)
        m.set("RV", rv)
        m.set_restart_numbers(p.P0, 0.0, 0)
        m.initialize()
    o.set_rk4_count(0)
    for name in ("update_rho", "update_p0", "update_particle", "update_rv_woq"):
        getattr(o, name)()
        getattr(s, name)(0)
    for f in ("RV_new", "RV_np1"):
        a, b = s.get(f), o.get(f)
        assert np.max(np.abs(a - b)) <= 1e-14 * np.max(np.abs(b)), (f, shape)
    o.close()
    s.close()
