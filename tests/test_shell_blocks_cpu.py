"""The quotient of the shell-block gather (div_rad in csrc/shell_blocks.h): two Newton steps from
a times the rounded 1 / r give the correctly rounded a / r, for the radii of the shell tables.
Restated here operation by operation, each FMA rounded once (exact rational arithmetic)."""
from fractions import Fraction

import numpy as np
import pytest


def _fma(a, b, c):
    v = Fraction(a) * Fraction(b) + Fraction(c)
    return v.numerator / v.denominator  # int / int rounds correctly


def _div_rad(a, r, y):
    q0 = a * y
    q1 = _fma(_fma(-q0, r, a), y, q0)
    return _fma(_fma(-q1, r, a), y, q1)


@pytest.mark.parametrize("seed", range(4))
def test_newton_quotient_is_the_division(seed):
    rng = np.random.default_rng(seed)
    r2 = rng.integers(1, 128 ** 2, 6000)
    # sums of Float32 terms: any sign, magnitudes from Float32's smallest to its largest
    a = rng.standard_normal(6000) * 2.0 ** rng.integers(-149, 128, 6000)
    a[:200] = np.float32(a[:200])
    a[200:300] = 0.0
    a[300:1500] = np.nextafter(np.sqrt(r2[300:1500]) * rng.integers(1, 2000, 1200), np.inf)
    for x, q in zip(a.tolist(), r2.tolist()):
        r = float(np.sqrt(float(q)))
        assert _div_rad(x, r, 1.0 / r) == x / r, (x, q)
