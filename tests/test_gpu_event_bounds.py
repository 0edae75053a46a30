"""The moves' folds around the vertex count where their form changes (2^19): real weights, runs of every
class, events at the highest positions, as a sweep returns them and through whole phases.  Below the
line a run is ordered by bits in LDS, which 2^19 vertices fill; above it the events are sorted and runs of
1024 and more folded by a wave each."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

SIZES = [2, 8, 9, 63, 64, 65, 66, 127, 128, 129, 500, 1023, 1024, 1025, 5000, 70000] + [70] * 300


def _stars(n, sizes, seed):
    """Stars whose centres have the smallest ids and whose leaves the largest; a path ties the rest."""
    rng = np.random.default_rng(seed)
    leaves = n - 1 - rng.permutation(int(np.sum(sizes)))
    pairs = np.stack([np.repeat(np.arange(len(sizes)), sizes), leaves], 1)
    rest = np.arange(len(sizes), n - len(leaves))
    pairs = np.concatenate([pairs, np.stack([rest[:-1], rest[1:]], 1)])
    w = np.concatenate([rng.uniform(0.5, 1.0, len(leaves)), rng.uniform(0.01, 0.1, len(rest) - 1)])
    return po.from_edge_list(n, pairs, w)


@pytest.mark.parametrize("n", [110003, (1 << 19) - 1, 1 << 19, (1 << 19) + 1, 600001])
def test_stars(ctx, n):
    g = _stars(n, SIZES, n)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = po.init_degrees(g)
    st = (np.arange(n), np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    t_o, cw_o, ds_o, dd_o = po.sweep(g, *st)
    assert np.sort(np.bincount(t_o[t_o != st[0]], minlength=n))[-1] == 70000
    t, cw, ds, dd = dg.sweep(*st)
    assert np.array_equal(t, t_o) and np.array_equal(ds, ds_o)
    assert np.array_equal(dd.view(np.uint64), dd_o.view(np.uint64))
    nc, colors = po.color(g, 4)
    for kw in (dict(), dict(mode="vorder", num_color=nc + 1, colors=colors), dict(mode="color", num_color=nc + 1, colors=colors)):
        q_o, cv_o, it_o = po.louvain_phase(g, **kw)
        q, cv, it = dg.louvain_phase(sequential=True, **kw)
        assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o), kw


@pytest.mark.parametrize("n", [8193, 100003, (1 << 20) - 1, 1 << 20, (1 << 20) + 1])
def test_random_moves(ctx, n):
    """The changes of a sweep on random rows, a few of them long, at the sizes where the sorts change."""
    rng = np.random.default_rng(n)
    d = rng.integers(0, 4, n)
    d[rng.choice(n, 50, replace=False)] = rng.choice([8, 20, 50, 100, 300, 600], 50)
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = po.init_degrees(g)
    st = (np.arange(n), np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    _, _, ds_o, dd_o = po.sweep(g, *st)
    _, _, ds, dd = dg.sweep(*st)
    assert np.array_equal(ds, ds_o)
    assert np.array_equal(dd.view(np.uint64), dd_o.view(np.uint64))


def test_time_of_many_long_runs(ctx):
    """Runs of 70 events are ordered by a workgroup each, at a cost that goes with the run: the scattering of
    seven thousand runs' events, times 13 (times 43 where each walked bits for all of the graph's vertices)."""
    n = 1 << 19
    g = _stars(n, [70] * 7000, 3)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    st = dg.phase_begin(thresh=-1.0)
    ctx.set_profiling(True)
    ctx.reset_stats()
    st.step()
    long, scatter = (ctx.kernel_stats(k)[2] for k in ("ev_fold_long", "ev_scatter"))
    ctx.set_profiling(False)
    st.end(want_cvect=False)
    assert 0 < long < 25 * scatter
