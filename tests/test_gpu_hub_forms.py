"""The hub rows' forms under the default tuning: in LDS by a workgroup around the sizes where its
tables change (512, 1024, 2048, 4096), longer rows of whole weights in one table, others sorted.
Targets and clusterWeights have the oracle's bits, also with self-loops, repeated tails, a giant
community, hubs frozen by early termination, and in a batch."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

N = 12000


def _graph(degs, whole, seed):
    rng = np.random.default_rng(seed)
    d = rng.integers(0, 6, N)
    hubs = 7 + 3 * np.arange(len(degs))
    d[hubs] = degs
    offs = np.concatenate([[0], np.cumsum(d)])
    tails = rng.integers(0, N, offs[-1])
    for h in hubs:
        own = offs[h] + rng.choice(d[h], 4, replace=False)
        tails[own[:h % 5]] = h
    w = rng.integers(0, 40, offs[-1]).astype(float) if whole else rng.uniform(0.1, 1.0, offs[-1])
    return po.make_graph(offs, tails, w), hubs, rng


SETS = {"lds": [512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 700, 3000],
        "with longer ones": [511, 512, 1500, 4096, 4097, 4098, 6143, 6144, 8191, 8193, 30000],
        "one": [512], "one long": [5000],
        "too many": [600] * 1600 + [1100, 5000, 6000]}


@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("name", list(SETS))
def test_sweeps(ctx, name, whole):
    g, hubs, rng = _graph(SETS[name], whole, len(name))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    # a phase, so that the hub rows' weights are looked at
    st = dg.phase_begin(thresh=-1.0)
    for it in range(4):
        st.sweep()
        s = st.state()
        t_o, cw_o, _, _ = po.sweep(g, s["curr"], s["csize"], s["cdeg"].copy(), s["vdeg"], s["constant"])
        assert np.array_equal(s["target"], t_o), it
        assert np.array_equal(s["cw"].view(np.uint64), cw_o.view(np.uint64)), it
        st.step()
    st.end(want_cvect=False)
    # a giant community that holds the hubs or not, halves, and few communities
    vdeg, c = po.init_degrees(g)
    ids = np.arange(N)
    giant = np.where(rng.random(N) < 0.7, 5, ids)
    for curr in (giant, np.where(np.isin(ids, hubs), ids, giant), ids % 2, ids % 61, ids // 40 * 40):
        a = (curr, np.bincount(curr, minlength=N), np.bincount(curr, vdeg, N), vdeg, c)
        t_o, cw_o, _, _ = po.sweep(g, *a)
        t, cw, _, _ = dg.sweep(*a)
        assert np.array_equal(t, t_o)
        assert np.array_equal(cw.view(np.uint64), cw_o.view(np.uint64))


@pytest.mark.parametrize("whole", [False, True])
def test_phases(ctx, whole):
    g, _, _ = _graph(SETS["with longer ones"], whole, 5)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    nc, colors = po.color(g, 4)
    for kw in (dict(), dict(mode="color", num_color=nc + 1, colors=colors), dict(et_type=2, et_delta=0.25), dict(et_type=1)):
        q_o, cv_o, it_o = po.louvain_phase(g, **kw)
        q, cv, it = dg.louvain_phase(sequential=True, **kw)
        assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o), kw


def test_batch(ctx):
    graphs = [_graph(SETS[k], w, 3)[0] for k in ("lds", "with longer ones") for w in (False, True)]
    dgs = [ctx.upload(vite_amd.CSR(g.offs, g.edges)) for g in graphs]
    batch = vite_amd.Batch(ctx, dgs)
    res, _ = batch.run(sequential=True)
    batch.free()
    for g, r in zip(graphs, res):
        o = po.run(g)
        assert r.call_q == o.call_q and r.call_iters == o.call_iters and r.level_nv == o.level_nv
