"""The stage kernels divide by 3 and 6 as q = x r, q + (x - D q) r with r the rounded reciprocal
and both steps fused (div_by in csrc/ptf_device.hpp).  That is the correctly rounded quotient:
here the same steps in exact rational arithmetic, rounded once each, against the exact quotient.
"""
from fractions import Fraction

import numpy as np
import pytest


def _round(x, T):
    """A rational rounded once to T (x within the normal range)."""
    if T is np.float64:
        return float(x)                     # Fraction -> float rounds correctly, ties to even
    if x == 0:
        return 0.0
    e = abs(x).numerator.bit_length() - abs(x).denominator.bit_length()
    for k in (e - 24, e - 23):              # 24 significant bits
        s = x / Fraction(2) ** k
        if 2 ** 23 <= abs(s) <= 2 ** 24:
            return float(Fraction(round(s)) * Fraction(2) ** k)
    raise AssertionError("scale")


@pytest.mark.parametrize("D", [3, 6])
@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_quotient_is_correctly_rounded(D, T):
    rng = np.random.default_rng(D)
    x = np.concatenate([rng.standard_normal(4000) * 10.0 ** rng.uniform(-25, 25, 4000),
                        np.arange(1, 200), np.nextafter(np.arange(1, 50) * 3.0, 0)]).astype(T)
    r = Fraction(_round(Fraction(1, D), T))
    for v in x:
        v = Fraction(float(v))
        q = Fraction(_round(v * r, T))
        rest = Fraction(_round(v - q * D, T))
        assert _round(rest * r + q, T) == _round(v / D, T)
