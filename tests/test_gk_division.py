"""The two-operation division of the Green-Kubo running means (div_by in gk.hip)."""
from fractions import Fraction

import numpy as np


def test_division_in_two_operations():
    """For c < 2^32 the quotient RN(a/c) is RN(a yh + RN(a yl)), in exact
    rationals with one rounding each."""
    rng = np.random.default_rng(3)
    for _ in range(2000):
        c = int(rng.integers(1, 2 ** int(rng.integers(1, 33))))
        a = float(rng.standard_normal() * 2.0 ** int(rng.integers(-300, 300)))
        yh = 1.0 / c
        yl = float(Fraction(1) - Fraction(c) * Fraction(yh)) / c
        q = float(Fraction(a) * Fraction(yh) + Fraction(a * yl))   # one rounding
        assert q == a / c, (a, c)
