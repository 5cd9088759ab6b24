"""Weight statistics of the setup report from uniform parts."""
import numpy as np
import pytest

from loopstructural_amd.interpolators import _weight_statistics


@pytest.mark.parametrize("parts", [
    [np.array([1.0, 2.0, 5.0])], [(0.1, 7)], [(0.1, 7), (0.3, 1)],
    [np.array([2.0]), (0.5, 4), np.array([0.1, 9.0])]])
def test_matches_the_arrays(parts):
    w = np.concatenate([p if isinstance(p, np.ndarray) else np.full(p[1], p[0]) for p in parts])
    mean, lo, hi = _weight_statistics(parts)
    assert lo == w.min() and hi == w.max()
    assert mean == pytest.approx(w.mean(), rel=1e-14)
