"""The comparison of partitions with few communities, where a few pairs hold most of the vertices: the
oracle's counts and floats at the edges of the counting's chunks, also where pairs share an LDS slot
(above a few thousand vertices, where the oracle's walk of all pairs would take minutes, numpy's counts of
the groups), and a counting time that does not grow as the communities get fewer."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _partitions(n, k, seed):
    rng = np.random.default_rng(seed)
    truth = np.minimum((k * rng.random(n) ** 1.5).astype(np.int64), k - 1)
    return truth, np.where(rng.random(n) < 0.15, rng.integers(0, k, n), truth)


def _expected(a, b):
    if len(a) < 5000:
        return po.compare(a, b)

    def inside(sizes):
        return int((sizes * (sizes - 1) // 2).sum())

    ss = inside(np.unique(a * (b.max() + 1) + b, return_counts=True)[1])
    sd, ds = inside(np.bincount(a)) - ss, inside(np.bincount(b)) - ss
    return dict(n=len(a), nc_truth=a.max() + 1, nc_found=b.max() + 1, same_same=ss, same_diff=sd, diff_same=ds,
                precision=ss / (ss + ds), recall=ss / (ss + sd))


@pytest.mark.parametrize("n", [255, 256, 257, 1023, 1025, 4097, 65537, 300007, 1024 * 1024 + 1, 2048 * 1024 + 1])
def test_few_communities(ctx, n):
    for k in (1, 2, 3, 40, 700):
        truth, found = _partitions(n, k, n + k)
        for a, b in ((truth, found), (found, truth), (truth, np.zeros(n, np.int64))):
            o = _expected(a, b)
            s = ctx.compare_communities(a, b)
            for key, v in o.items():
                assert s[key] == v or (np.isnan(s[key]) and np.isnan(v)), (k, key)


def test_counting_time_with_few_communities(ctx):
    n, us = 1000003, {}
    for k in (2, 1024):
        truth, found = _partitions(n, k, k)
        best = np.inf
        for _ in range(5):
            ctx.set_profiling(True)
            ctx.reset_stats()
            ctx.compare_communities(truth, found)
            best = min(best, ctx.kernel_stats("cmp_count")[2])
            ctx.set_profiling(False)
        us[k] = 1e3 * best
    # one atomic per vertex on four lines of memory took 25 times as long as on a thousand communities'
    assert us[2] < 4 * us[1024], us


@pytest.mark.parametrize("n", [70001, 300007])
def test_singletons(ctx, n):
    """As many communities as vertices: the sizes' host loop at its longest."""
    rng = np.random.default_rng(n)
    ids, half = rng.permutation(n), np.arange(n) // 2
    for a, b in ((ids, ids), (ids, half), (half, ids)):
        s = ctx.compare_communities(a, b)
        pairs = {True: n // 2, False: 0}
        assert s["same_same"] == 0
        assert (s["same_diff"], s["diff_same"]) == (pairs[a is half], pairs[b is half])
        for part, gini in ((a, s["gini_truth"]), (b, s["gini_found"])):
            size = np.sort(np.bincount(part)).astype(float)
            k = len(size)
            num = float(((np.arange(k) + 1) * size).sum())  # whole numbers below 2^53
            assert gini == (2 * num) / (k * size.sum()) - (k + 1.0) / k
