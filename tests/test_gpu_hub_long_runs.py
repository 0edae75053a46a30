"""Hub rows whose neighbours lie in a few communities: runs of hundreds to thousands of entries, many of
about one length or one among short ones, of real and of whole weights.  Targets and clusterWeights have
the oracle's bits, and the runs' time does not grow as they fall into fewer waves."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

N = 20000


def _graph(hubs, length, whole):
    rng = np.random.default_rng(hubs + length)
    d = rng.integers(0, 5, N)
    d[rng.choice(N, hubs, replace=False)] = length + rng.integers(0, length // 8, hubs)
    offs = np.concatenate([[0], np.cumsum(d)])
    w = rng.integers(1, 9, offs[-1]).astype(float) if whole else rng.uniform(0.1, 1.0, offs[-1])
    return po.make_graph(offs, rng.integers(0, N, offs[-1]), w), rng


def _states(g, rng, counts):
    vdeg, c = po.init_degrees(g)
    for k in counts:
        curr = rng.integers(0, k, N)
        yield k, (curr, np.bincount(curr, minlength=N), np.bincount(curr, vdeg, N), vdeg, c)


@pytest.fixture(params=[0, 1 << 30], ids=["workgroup per hub", "flat"])
def form(ctx, request):
    keep = ctx.tuning
    ctx.set_tuning(hub_block_min=request.param)
    yield request.param
    ctx.set_tuning(**keep)


@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("hubs,length", [(3, 9000), (40, 9000), (30, 26000)])
def test_few_communities(ctx, form, hubs, length, whole):
    g, rng = _graph(hubs, length, whole)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    counts = [1, 2, 3, 10, 24, 25, 36, 100] if length < 20000 else [2, 3]
    for k, st in _states(g, rng, counts):
        t_o, cw_o, _, _ = po.sweep(g, *st)
        t, cw, _, _ = dg.sweep(*st)
        assert np.array_equal(t, t_o), k
        assert np.array_equal(cw.view(np.uint64), cw_o.view(np.uint64)), k


def test_one_giant_among_single_entries(ctx, form):
    g, rng = _graph(40, 9000, False)
    vdeg, c = po.init_degrees(g)
    curr = np.where(rng.random(N) < 0.5, 3, np.arange(N))
    st = (curr, np.bincount(curr, minlength=N), np.bincount(curr, vdeg, N), vdeg, c)
    t_o, cw_o, _, _ = po.sweep(g, *st)
    t, cw, _, _ = ctx.upload(vite_amd.CSR(g.offs, g.edges)).sweep(*st)
    assert np.array_equal(t, t_o) and np.array_equal(cw.view(np.uint64), cw_o.view(np.uint64))


def test_time_of_many_long_runs(ctx):
    """640 runs of about 900 real weights, 64 to a wave: their lanes fold them side by side, as they
    fold runs of 90 (the wave folding one after another took 25 times as long as those)."""
    keep = ctx.tuning
    ctx.set_tuning(hub_block_min=1 << 30)
    try:
        g, rng = _graph(64, 9000, False)
        dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
        best = {}
        for k, st in _states(g, rng, [100, 10]):
            for _ in range(4):
                ctx.set_profiling(True)
                ctx.reset_stats()
                dg.sweep(*st)
                best[k] = min(best.get(k, np.inf), ctx.kernel_stats("hub_runs")[2])
                ctx.set_profiling(False)
        assert 0 < best[10] < 12 * best[100], best
    finally:
        ctx.set_tuning(**keep)
