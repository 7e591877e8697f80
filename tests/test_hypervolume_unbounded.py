"""The hypervolume of a set with a point at minus infinity in one coordinate is
infinite, whatever coordinates the others share with it."""
import numpy as np
import pytest


@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 6])
def test_one_unbounded_point(cdp, d):
    rng = np.random.default_rng(d)
    for _ in range(300):
        n = int(rng.integers(1, 8))
        pts = rng.integers(0, 4, (n, d)) / 4.0
        pts[int(rng.integers(0, n)), int(rng.integers(0, d))] = -np.inf
        assert cdp.hypervolume(pts) == np.inf, pts.tolist()
