"""The packed first Poisson pass with two row sets a block (8 rows a set and x
lengths from 128 on) against the five passes (TPX_FFT_PASSES=5) in the coefficient
solve: the same operations up to the order of the transforms' sums, so the same
iterations and results within 1e-12.  The y lengths 64 and 128 are the two that
give 8 rows."""
import numpy as np
import pytest

from test_gpu_coef_three_pass import _case, _solver

pytestmark = pytest.mark.gpu

SHAPES = [(16, 64, 128), (64, 128, 128), (16, 128, 256), (16, 64, 512)]


@pytest.mark.parametrize("shape", SHAPES)
def test_coefficient_solve_equals_five_pass(gpu_available, monkeypatch, shape):
    p, C, RHS, P0 = _case(shape)
    out = []
    for passes in ("3", "5"):
        s = _solver(p, monkeypatch, passes)
        out.append(s.poisson_solve(C, P0, RHS))
        s.close()
    (P3, i3), (P5, i5) = out
    assert i3 == i5 > 2
    assert np.max(np.abs(P3 - P5)) <= 1e-12 * np.max(np.abs(P5))
