"""The cosines written out in the transform kernels (the 16- and 32-point
twiddles, cos(q pi/16)) are the doubles nearest to their values, worked out
here in whole numbers to 60 digits."""
import os
import re
from fractions import Fraction

from conftest import PKG

SCALE = 10 ** 60


def _atan_inv(n):
    """SCALE atan(1/n), by its series."""
    term, total, k = SCALE // n, 0, 0
    while term:
        total += (-1) ** k * term // (2 * k + 1)
        term //= n * n
        k += 1
    return total


PI = 4 * (4 * _atan_inv(5) - _atan_inv(239))  # Machin's formula


def _cos(q):
    """cos(q pi/16) as a fraction, by its series."""
    x2 = (q * PI // 16) ** 2 // SCALE
    term, total, k = SCALE, 0, 0
    while term:
        total += (-1) ** k * term
        k += 1
        term = term * x2 // SCALE // ((2 * k - 1) * (2 * k))
    return Fraction(total, SCALE)


def test_written_out_cosines_are_the_nearest_doubles():
    with open(os.path.join(PKG, "csrc", "k_fft.hip")) as f:
        text = re.sub(r"//.*", "", f.read())
    found = re.findall(r"\b0\.\d{12,}\b", text)
    exact = [_cos(q) for q in range(8)]
    nearest = [float(e) for e in exact]  # a fraction's float is correctly rounded
    assert len(found) >= 10, found
    for s in found:
        q = min(range(8), key=lambda k: abs(Fraction(s) - exact[k]))
        assert float(s) == nearest[q], f"{s}: cos({q} pi/16) is {nearest[q]!r}"
