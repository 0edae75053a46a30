"""The comparison where every vertex has a pair of its own, where all share one, and between: the
oracle's counts and floats."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 255, 257, 1000, 3001])
def test_pairs(ctx, n):
    rng = np.random.default_rng(n)
    ids = np.arange(n)
    zero = np.zeros(n, np.int64)
    some = rng.integers(0, max(1, n // 7), n)
    sparse = rng.integers(0, 5, n) * 1000003  # far ids, most of them of no vertex
    for truth, found in ((ids, zero), (zero, ids), (zero, zero), (ids, ids[::-1].copy()), (some, ids % 3), (some, some),
                         (some, np.where(rng.random(n) < 0.1, 0, some)), (sparse, some)):
        o = po.compare(truth, found)
        s = ctx.compare_communities(truth, found)
        for k, v in o.items():
            assert s[k] == v or (np.isnan(s[k]) and np.isnan(v)), k
