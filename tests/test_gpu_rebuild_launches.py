"""A rebuild of more than 8192 vertices with overflowing communities: one launch for both totals and both
largest rows, the second time the rows alone, and no launch for long runs where no community can hold
one.  The coarse graph has the oracle's bytes."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entries,long_runs", [(3, False), (40, True)])
def test_overflow_launches(ctx, entries, long_runs):
    n, rng = 20000, np.random.default_rng(entries)
    d = np.full(n, entries)
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    part = np.arange(n) // 50 * 50  # 150 or 2000 entries a community, most of communities of their own
    ctx.set_profiling(True)
    ctx.reset_stats()
    r = dg.rebuild(part)
    n_of = {k: ctx.kernel_stats(k)[1] for k in ("rb_totals", "max_degree", "rb_fold", "rb_fold_long")}
    ctx.set_profiling(False)
    assert n_of == dict(rb_totals=2, max_degree=0, rb_fold=1, rb_fold_long=int(long_runs))
    a, b = r.download(), po.rebuild(g, part)
    assert np.array_equal(a.offs, b.offs) and np.array_equal(a.edges.view(np.uint8), b.edges.view(np.uint8))
    # the largest row the rebuild found is the one that later launches rely on
    st = r.phase_begin(thresh=-1.0, sequential=True)
    st.sweep()
    s = st.state()
    st.end(want_cvect=False)
    vdeg, c = po.init_degrees(b)
    t_o, _, _, _ = po.sweep(b, np.arange(b.nv), np.ones(b.nv, np.int64), vdeg.copy(), vdeg, c)
    assert np.array_equal(s["target"], t_o)
