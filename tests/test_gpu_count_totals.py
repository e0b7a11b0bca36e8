"""The particle advance adds to the totals of the scan's blocks (4096 cells each)
while it counts the cells: two coupled, heated steps against the oracle on grids
below one block, of exactly one, of two and of many, with few particles, and
with several in every cell; and particles that cross between the blocks."""
import numpy as np
import pytest

from test_gpu_parity import TOL_1, oracle_from_case, solver_from_case, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cell", [0.02, 3.0])
@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 16, 16), (32, 16, 16), (32, 64, 32)])
def test_counted_totals_match_the_oracle(gpu_available, shape, per_cell):
    from tpx import ic
    nz, ny, nx = shape
    npart = int(nx * ny * nz * per_cell) + 1
    case = ic.make_case(nx, npart, nu=0.05, seed=9, St=1.0, phi=0.3, heat=True, drag_limit=True, shape=shape)
    rng = np.random.default_rng(3)
    for q in "uvw":  # about half a cell a step
        case.particles[q] += 0.5 * case.params.Lx / nx / case.params.dt * rng.standard_normal(npart)
    o, s = oracle_from_case(case), solver_from_case(case)
    o.step(2)
    s.step(2)
    e = state_errors(o, s, case)
    assert max(e.values()) <= TOL_1, e
