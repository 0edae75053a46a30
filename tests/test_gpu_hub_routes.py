"""Which hub rows take the table of whole weights: a few long ones beside many that go to LDS, and not the
long rows of a dense graph, nor long ones alone, whose sweeps the sort serves better.  Targets and
clusterWeights have the oracle's bits on every route."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _graph(n, long, mid, seed, whole=True):
    rng = np.random.default_rng(seed)
    d = rng.integers(0, 6, n)
    hubs = rng.permutation(n)[:len(long) + len(mid)]
    d[hubs] = list(long) + list(mid)
    offs = np.concatenate([[0], np.cumsum(d)])
    tails = rng.integers(0, n, offs[-1])
    for h in hubs[::3]:
        tails[offs[h] + rng.choice(d[h], 4, replace=False)] = h
    w = rng.integers(0, 40, offs[-1]).astype(float) if whole else rng.uniform(0.1, 1.0, offs[-1])
    return po.make_graph(offs, tails, w)


LONG = [4097, 4098, 6143, 6144, 8191, 8193, 30000]
MID = [512, 513, 700, 1024, 1025, 2048, 4095, 4096] * 7
# rows, whether the table serves them; the last: more than 2^20 entries and no row with much of them
CASES = {"few beside many": (LONG, MID, True), "one too many": (LONG + [5000], MID, False), "alone": (LONG, [], False),
         "dense": ([4500] * 300, [4000] * 300, False), "many entries": ([8000] * 140, [600] * 1120, False),
         "a giant among them": ([8000] * 130 + [70000], [600] * 1120, True)}


@pytest.mark.parametrize("n", [8000, 9000])  # the set-up in one workgroup, and in launches
@pytest.mark.parametrize("name", list(CASES))
def test_routes(ctx, n, name):
    long, mid, table = CASES[name]
    g = _graph(n, long, mid, n + len(name))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    st = dg.phase_begin(thresh=-1.0)
    for it in range(3):
        ctx.set_profiling(True)
        ctx.reset_stats()
        st.sweep()
        used = ctx.kernel_stats("hubw_insert")[1]
        ctx.set_profiling(False)
        assert used == (1 if table else 0)
        s = st.state()
        t_o, cw_o, _, _ = po.sweep(g, s["curr"], s["csize"], s["cdeg"].copy(), s["vdeg"], s["constant"])
        assert np.array_equal(s["target"], t_o), it
        assert np.array_equal(s["cw"].view(np.uint64), cw_o.view(np.uint64)), it
        st.step()
    st.end(want_cvect=False)


def test_phases(ctx):
    g = _graph(12000, LONG, MID, 5)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    nc, colors = po.color(g, 4)
    for kw in (dict(), dict(mode="color", num_color=nc + 1, colors=colors), dict(et_type=2, et_delta=0.25), dict(et_type=1)):
        q_o, cv_o, it_o = po.louvain_phase(g, **kw)
        q, cv, it = dg.louvain_phase(sequential=True, **kw)
        assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o), kw


def test_gains_of_few_hubs_with_many_communities(ctx):
    """Sixteen hubs with a community per entry: forming the gains may not take a multiple of the adding."""
    g = _graph(20000, [10000] * 16, [560] * 128, 3)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    st = dg.phase_begin(thresh=-1.0)
    best = {}
    for _ in range(5):
        ctx.set_profiling(True)
        ctx.reset_stats()
        st.sweep()
        for k in ("hubw_insert", "hubw_gain"):
            best[k] = min(best.get(k, np.inf), ctx.kernel_stats(k)[2])
        ctx.set_profiling(False)
    st.end(want_cvect=False)
    # an atomic per wave and hub on one line of memory took 11 times as long
    assert 0 < best["hubw_gain"] < 3 * best["hubw_insert"], best


@pytest.mark.parametrize("n", [8000, 9000])
@pytest.mark.parametrize("rows,lds", [([1500] * 1023, True), ([1500] * 1024, False), ([600] * 1024 + [1500] * 400, True)])
def test_many_rows_in_lds(ctx, n, rows, lds):
    """Rows that go to LDS, up to a thousand of any length, more where they are short on average."""
    g = _graph(n, [], rows, n + len(rows), whole=False)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    st = dg.phase_begin(thresh=-1.0)
    for it in range(2):
        ctx.set_profiling(True)
        ctx.reset_stats()
        st.sweep()
        used = ctx.kernel_stats("local_move_hub_sort")[1]
        ctx.set_profiling(False)
        assert used == (0 if lds else 1)
        s = st.state()
        t_o, cw_o, _, _ = po.sweep(g, s["curr"], s["csize"], s["cdeg"].copy(), s["vdeg"], s["constant"])
        assert np.array_equal(s["target"], t_o), it
        assert np.array_equal(s["cw"].view(np.uint64), cw_o.view(np.uint64)), it
        st.step()
    st.end(want_cvect=False)
