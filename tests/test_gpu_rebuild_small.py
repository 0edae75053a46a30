"""Rebuilds of graphs around the size where one workgroup lists the members and scans the rows,
and communities around the numbers of distinct neighbours that the table holds.  The coarse
CSR equals the oracle's byte for byte."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _same(ctx, g, part):
    r, r_o = ctx.upload(vite_amd.CSR(g.offs, g.edges)).rebuild(part).download(), po.rebuild(g, part)
    assert np.array_equal(r.offs, r_o.offs)
    assert np.array_equal(r.edges.view(np.uint8), r_o.edges.view(np.uint8))


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 1000, 1024, 1025, 4097, 8191, 8192, 8193])
def test_sizes(ctx, n):
    rng = np.random.default_rng(n)
    d = rng.integers(0, 9, n)
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
    for part in (np.arange(n), np.zeros(n, np.int64), np.arange(n)[::-1].copy(), rng.integers(0, n, n),
                 rng.integers(0, max(1, n // 9), n) * 8, np.arange(n) // 70 * 70):
        _same(ctx, g, part.astype(np.int64))


@pytest.mark.parametrize("n", [6000, 9000])
def test_distinct_neighbours(ctx, n):
    """Communities with 1 to 1100 neighbours: the first of its three members has most of the row."""
    rng = np.random.default_rng(n)
    keys = [1, 64, 100, 127, 128, 129, 130, 191, 192, 193, 255, 256, 257, 300, 500, 511, 512, 513, 514, 575, 576, 577, 800, 1100]
    d = np.zeros(n, np.int64)
    tails = [[] for _ in range(n)]
    for i, k in enumerate(keys):
        far = 200 + rng.choice(n - 200, k, replace=False)
        far = np.concatenate([far, rng.choice(far, k // 2), [3 * i + 1] * (i % 3)])  # repeats, and inner entries
        rng.shuffle(far)
        cut = len(far) * 2 // 3
        tails[3 * i], tails[3 * i + 1] = list(far[:cut]), list(far[cut:])
    d = np.array([len(x) for x in tails])
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, np.concatenate([np.array(x, np.int64) for x in tails]), rng.uniform(0.1, 1.0, offs[-1]))
    part = np.arange(n)
    for i in range(len(keys)):
        part[3 * i:3 * i + 3] = 3 * i + 2
    _same(ctx, g, part)
    _same(ctx, g, n - 1 - part)


@pytest.mark.parametrize("n", [50, 8192, 8193])
def test_ids_out_of_range_are_counted(ctx, n):
    g = ctx.gen_rgg(5, n)
    part = np.arange(n)
    part[[0, 7, n - 1]] = [-1, n, n + 5]
    with pytest.raises(vite_amd.VtError, match="3 community ids outside"):
        g.rebuild(part)
    assert g.rebuild(np.arange(n)).nv == n
