"""The sliced path's quotient by a row's temperature (one product by the
rounded reciprocal, one correction by the exact remainder) is the IEEE
quotient that sampling.py:88 computes, in exact rational arithmetic."""
from fractions import Fraction

import numpy as np


def quotient(a: float, t: float) -> float:
    inv = 1.0 / t
    q = a * inv
    rem = float(Fraction(a) - Fraction(q) * Fraction(t))   # fma(-q, t, a): float(Fraction) rounds to nearest even
    return float(Fraction(rem) * Fraction(inv) + Fraction(q))


def test_quotients_are_ieee():
    rng = np.random.default_rng(1)
    temperatures = [0.1, 0.3, 0.7, 0.9, 1.0, 1.1, 1.3, 1.7, 3.0, 49.0, 99.9, 1e-3, 1e-9, np.nextafter(1.0, 2.0),
                    np.nextafter(1.0, 0.0), np.nextafter(2.0, 0.0)] + list(rng.uniform(0.01, 100, 40))
    differ_from_product = 0
    for t in map(float, temperatures):
        floats = -np.abs(rng.normal(0, 20, 200).astype(np.float32).astype(np.float64))
        tiny = -np.ldexp(rng.uniform(1, 2, 40).astype(np.float32).astype(np.float64), rng.integers(-140, 30, 40))
        for a in map(float, np.concatenate([floats, -np.abs(rng.normal(0, 20, 100)), tiny, [0.0]])):
            assert quotient(a, t) == a / t, (a, t)
            differ_from_product += a * (1.0 / t) != a / t
    assert differ_from_product > 1000
