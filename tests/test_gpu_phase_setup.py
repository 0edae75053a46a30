"""The set-up of a phase around the size where one workgroup does it: degrees, 1/2m, state and
sweep lists as the separate launches form them (a sweep reaches every vertex through its list)."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _graph(n, seed):
    """Rows of every bucket, in no order, some of them hubs."""
    rng = np.random.default_rng(seed)
    d = rng.choice([0, 1, 7, 8, 15, 16, 31, 32, 63, 64, 127, 128, 191, 255, 256, 511, 512, 700, 1023, 1024, 1500], n,
                   p=[0.05] + [0.1] * 9 + [0.05 / 11] * 11)
    offs = np.concatenate([[0], np.cumsum(d)])
    return po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))


@pytest.mark.parametrize("et", [0, 2])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 1023, 1024, 1025, 3000, 8191, 8192, 8193])
def test_setup(ctx, n, et):
    g = _graph(n, n)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    vdeg, c = dg.init_degrees()
    assert np.array_equal(vdeg, po.init_degrees(g)[0])
    if not vdeg.sum() > 0.0:
        return
    st = dg.phase_begin(thresh=-1.0, et_type=et, et_delta=0.25)
    s = st.state()
    ids = np.arange(n)
    assert np.array_equal(s["curr"], ids) and np.array_equal(s["csize"], np.ones(n))
    assert np.array_equal(s["vdeg"], vdeg) and np.array_equal(s["cdeg"], vdeg) and s["constant"] == c
    st.sweep()
    s = st.state()
    st.end(want_cvect=False)
    t_o, cw_o, _, _ = po.sweep(g, ids, np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    assert np.array_equal(s["target"], t_o)
    assert np.array_equal(s["cw"].view(np.uint64), cw_o.view(np.uint64))
