"""The quotient t / N by the reciprocal of a constant N (div_by in
pst_device.hpp): restated in exact rational arithmetic, rounded where the
kernel rounds, it is the correctly rounded quotient."""
from fractions import Fraction

import numpy as np
import pytest


@pytest.mark.parametrize("n", [3, 5, 6, 7])
def test_reciprocal_quotient_is_the_division(n):
    rng = np.random.default_rng(n)
    t = np.concatenate([
        np.ldexp(rng.uniform(1.0, 2.0, 4000), rng.integers(-900, 4, 4000)),
        np.ldexp(1.0 + rng.integers(0, 64, 500) * 2.0 ** -52, rng.integers(-60, 4, 500)),  # next to powers of two
        np.arange(1.0, 200.0) * n, np.nextafter(np.arange(1.0, 200.0) * n, 0.0),           # next to multiples of n
        [0.0],
    ])
    r = 1.0 / n
    for v in t.tolist():
        q = v * r
        rem = float(Fraction(v) - n * Fraction(q))
        assert float(Fraction(q) + Fraction(rem) * Fraction(r)) == v / n
