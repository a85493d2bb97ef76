"""The 2D sampler's division by a spacing in five operations equals the correctly rounded
quotient (exact rational arithmetic, so that no rounding of the check itself enters)."""
from fractions import Fraction

import numpy as np
import pytest


def _rn(x: Fraction) -> Fraction:
    """Round to float32's nearest, ties to even (normal range)."""
    if x == 0:
        return x
    e = 0
    a = abs(x)
    e = a.numerator.bit_length() - a.denominator.bit_length()
    if Fraction(2) ** e > a:
        e -= 1
    ulp = Fraction(2) ** (e - 23)
    return round(x / ulp) * ulp


def _refined(x: Fraction, s: Fraction):
    inv = _rn(1 / s)
    q = _rn(x * inv)
    q = _rn(q + _rn(x - q * s) * inv)
    r = x - q * s
    assert _rn(r) == r              # the second residual is exact
    return _rn(q + r * inv)


@pytest.mark.parametrize("seed", [0, 1])
def test_refined_division_is_correctly_rounded(seed):
    rng = np.random.default_rng(seed)
    ends = [1 << 23, (1 << 23) + 1, (1 << 24) - 1, (1 << 24) - 2, 11863283, 11863284]  # around 1, 2 and sqrt(2)
    ms = [int(v) for v in rng.integers(1 << 23, 1 << 24, 3000)]
    mx = [int(v) for v in rng.integers(1 << 23, 1 << 24, 3000)]
    pairs = list(zip(mx, ms)) + [(a, b) for a in ends for b in ends]
    # quotients next to a midpoint of two floats: x = round(s (2k + 1) / 2^25) for odd halves
    for b in ms[:1000]:
        half = (int(rng.integers(1 << 23, 1 << 24)) << 1) | 1
        a = (b * half) >> 24
        while a >= 1 << 24:
            a >>= 1
        if a >= 1 << 23:
            pairs += [(a, b), (a + 1 if a + 1 < 1 << 24 else a, b)]
    for a, b in pairs:
        x, s = Fraction(a, 1 << 20), Fraction(b, 1 << 23)
        assert _refined(x, s) == _rn(x / s), (a, b)
