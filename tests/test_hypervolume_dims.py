"""The hypervolume at every count of coordinates and at the smallest sets,
against inclusion-exclusion in rationals: one rounding per operation of a sum
of at most a few hundred terms below 1."""
import itertools
from fractions import Fraction

import numpy as np
import pytest


def exact(pts):
    total = Fraction(0)
    for r in range(1, len(pts) + 1):
        for sub in itertools.combinations(range(len(pts)), r):
            v = Fraction(1)
            for x in pts[list(sub)].max(0):
                v *= max(Fraction(0), 1 - Fraction(float(x)))
            total += v if r % 2 else -v
    return float(total)


@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 6, 7, 16])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 8])
def test_dims(cdp, d, n):
    rng = np.random.default_rng([d, n])
    for step in (0, 2, 4):  # continuous, and on grids: equal coordinates and equal points
        pts = rng.random((n, d)) if not step else rng.integers(0, step + 1, (n, d)) / step
        assert abs(cdp.hypervolume(pts) - exact(pts)) <= 1e-13
