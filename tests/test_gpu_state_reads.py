"""A phase's state and a sweep's results as a caller reads them: 64-bit ids and sizes, with the oracle's
values, and no launch or device memory for the widening."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 30, 8193, 300007])
def test_state(ctx, n):
    rng = np.random.default_rng(n)
    d = rng.integers(0, 5, n)
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = po.init_degrees(g)
    ids = np.arange(n)
    st = dg.phase_begin(thresh=-1.0, sequential=True)
    st.sweep()
    s = st.state()
    ctx.set_profiling(True)
    ctx.reset_stats()
    s = st.state()
    launches = ctx.kernel_stats("widen_ids")[1]
    ctx.set_profiling(False)
    st.end(want_cvect=False)
    assert launches == 0
    assert all(s[k].dtype == np.int64 for k in ("curr", "csize", "target"))
    assert np.array_equal(s["curr"], ids) and np.array_equal(s["csize"], np.ones(n, np.int64))
    if offs[-1] == 0:
        return
    t_o, cw_o, ds_o, _ = po.sweep(g, ids, np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    assert np.array_equal(s["target"], t_o) and np.array_equal(s["cw"].view(np.uint64), cw_o.view(np.uint64))
    t, _, ds, _ = dg.sweep(ids, np.ones(n, np.int64), vdeg, vdeg, c)
    assert np.array_equal(t, t_o) and np.array_equal(ds, ds_o) and ds.dtype == np.int64
