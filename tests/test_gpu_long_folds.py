"""Long left folds: vertex degrees, and a hub's counters, by a thread, a wave or a workgroup by
their length, side by side where every term is a whole number and in order otherwise.  All have
the bits of the oracle's in-order folds, also where whole numbers are too large for exact sums,
where a fraction comes late, and with negative weights and signed zeros."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

N = 6000


def _weights(kind, n, rng):
    w = rng.integers(1, 50, n).astype(float)
    if kind == "real":
        return rng.uniform(0.1, 1.0, n)
    if kind == "late":  # one fraction near the end
        w[-3] = 0.1
    if kind == "large":  # partial sums pass 2^53
        w = np.ldexp(w + rng.integers(0, 2, n) * 2.0 ** -40, 45)
    if kind == "signed":
        w = rng.integers(-50, 50, n).astype(float)
        w[::7] = -0.0
    return w


def _graph(deg, kind, seed):
    """A directed multigraph: vertex 3 has a row of `deg` entries (self-loops and repeated tails
    among them), ten more have rows around the lengths where the folds change, the rest are short."""
    rng = np.random.default_rng(seed)
    d = rng.integers(0, 6, N)
    d[3] = deg
    d[10:20] = [63, 64, 255, 256, 257, 511, 512, 513, 1024, 1025]
    offs = np.concatenate([[0], np.cumsum(d)])
    tails = rng.integers(0, N, offs[-1])
    own = offs[3] + rng.choice(deg, 5, replace=False)
    tails[own] = 3
    w = np.concatenate([_weights(kind, k, rng) if k > 20 else rng.integers(1, 9, k).astype(float) for k in d])
    return po.make_graph(offs, tails, w), rng


@pytest.mark.parametrize("kind", ["whole", "real", "late", "large", "signed"])
@pytest.mark.parametrize("deg", [1500, 8191, 8192, 8193, 40000])
def test_long_folds(ctx, deg, kind):
    g, rng = _graph(deg, kind, deg)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = po.init_degrees(g)
    v, _ = dg.init_degrees()
    assert np.array_equal(v.view(np.uint64), vdeg.view(np.uint64))
    # a community with most of the vertices: the hub's own, another's, or none
    giant = np.where(rng.random(N) < 0.7, 5, np.arange(N))
    halves = np.where(np.arange(N) % 2, 5, 8)
    for curr in (np.where(np.arange(N) == 3, 5, giant), np.where(np.arange(N) == 3, 3, giant), halves, np.arange(N)):
        size = np.bincount(curr, minlength=N)
        st = (curr, size, np.bincount(curr, vdeg, N), vdeg, c)
        t_o, cw_o, _, _ = po.sweep(g, *st)
        for hub_block_min in (0, 1 << 30):  # a workgroup per hub, and the flat launches
            keep = ctx.tuning
            ctx.set_tuning(hub_block_min=hub_block_min)
            try:
                t, cw, _, _ = dg.sweep(*st)
            finally:
                ctx.set_tuning(**keep)
            assert np.array_equal(t, t_o)
            assert np.array_equal(cw.view(np.uint64), cw_o.view(np.uint64))
