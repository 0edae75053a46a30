"""The end of an iteration: the moves folded into the communities and the modularity.  Three
forms by vertex count (one workgroup up to 8192 vertices, atomics up to 2^19, a sort above), and
in each the event runs take different folds by their length; all give the bits of the oracle's
in-order folds, and the modularity the bits of vt_modularity on the same arrays."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _stars(n, sizes, seed):
    """Stars of the given leaf counts whose centres have the smallest ids (two lone vertices
    join into the smaller id, so every leaf moves to its centre: runs of about that many
    events); the remaining vertices form a path."""
    rng = np.random.default_rng(seed)
    ids = len(sizes) + rng.permutation(n - len(sizes))
    pairs, w, k = [], [], 0
    for centre, s in enumerate(sizes):
        pairs += [(centre, v) for v in ids[k:k + s]]
        w.append(rng.uniform(0.5, 1.0, s))
        k += s
    rest = ids[k:]
    pairs += list(zip(rest[:-1], rest[1:]))
    w.append(rng.uniform(0.01, 0.1, max(0, len(rest) - 1)))
    return po.from_edge_list(n, np.sort(np.array(pairs), axis=1), np.concatenate(w))


SIZES = [2, 4, 7, 8, 9, 11, 12, 13, 23, 24, 25, 31, 32, 33, 60, 63, 64, 65, 100, 127, 128, 129, 500, 1023, 1024]
CASES = [(8191, SIZES), (8192, SIZES + [3000]), (8193, SIZES + [3000]), (14000, SIZES + [4095, 4096]),
         (20001, SIZES + [4097, 9000])]


@pytest.mark.parametrize("n,sizes", CASES, ids=[str(c[0]) for c in CASES])
def test_event_runs_of_every_length(ctx, n, sizes):
    g = _stars(n, sizes, n)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = po.init_degrees(g)
    st = (np.arange(n), np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    t_o, cw_o, ds_o, dd_o = po.sweep(g, *st)
    assert np.array_equal(np.sort(np.bincount(t_o[t_o != st[0]], minlength=n))[-5:], np.sort(sizes)[-5:])
    t, cw, ds, dd = dg.sweep(*st)
    assert np.array_equal(t, t_o)
    assert np.array_equal(ds, ds_o)
    assert np.array_equal(dd.view(np.uint64), dd_o.view(np.uint64))
    nc, colors = po.color(g, 4)
    for kw in (dict(), dict(mode="color", num_color=nc + 1, colors=colors), dict(et_type=2, et_delta=0.25),
               dict(mode="vorder", num_color=nc + 1, colors=colors)):
        q_o, cv_o, it_o = po.louvain_phase(g, **kw)
        q, cv, it = dg.louvain_phase(sequential=True, **kw)
        assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o), kw


@pytest.mark.parametrize("n", [20, 255, 1024, 1025, 2049, 5000, 8192, 8193, 30000])
@pytest.mark.parametrize("et", [0, 2])
def test_modularity_has_the_tree_sums_bits(ctx, n, et):
    dg = ctx.gen_rgg(n, n, 1.0)
    st = dg.phase_begin(thresh=-1.0, et_type=et, et_delta=0.25)
    for _ in range(3):
        q, _ = st.step()
        s = st.state()
        assert q == ctx.modularity(s["cw"], s["cdeg"], s["constant"])
    st.end(want_cvect=False)
