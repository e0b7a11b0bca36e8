"""A solve of the caller's system that stops after fewer iterations than the
last one took must not have queued that many: at most 4 beyond those that ran.
Such a solve expects the count of the one before, so a cold solve and then one
from its result are alternated; the iterations queued are the launches of the
transform's first pass that the kernel timing counts.  Three-pass and (an axis
of 8) five-pass form."""
import numpy as np
import pytest

from test_oracle_poisson_coef import manufactured

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 16, 64), (16, 8, 64)])
def test_iterations_queued_beyond_the_stop(gpu_available, shape):
    from tpx import Solver
    p, _, C, RHS = manufactured(shape, seed=sum(shape), spread=0.5)
    p.epsilon, p.Iteration1, p.Iteration2 = 1e-10, 50, 50
    s = Solver(p, np_capacity=1)
    s.timing(True)
    seen, P, its = 0, np.zeros(shape), []
    for warm in (False, True, False, True):
        P, n = s.poisson_solve(C, P if warm else np.zeros(shape), RHS)
        queued = s.timing_read()[1]["fft"] - seen
        seen += queued
        its.append(n)
        print(shape, "warm" if warm else "cold", "iterations", n, "queued", queued)
        assert n <= queued <= n + 4
    s.close()
    assert its[0] == its[2] > 4 and its[1] == its[3] < its[0] - 4, its
