"""Rebuilds and sweeps at the size where the vertex sorts change (2^20): members in vertex order and
every vertex in its sweep list, against the oracle."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8193, 100003, (1 << 20) - 1, 1 << 20, (1 << 20) + 1])
def test_vertex_sorts(ctx, n):
    rng = np.random.default_rng(n)
    d = rng.integers(0, 4, n)
    d[rng.choice(n, 50, replace=False)] = rng.choice([8, 20, 50, 100, 300, 600], 50)
    offs = np.concatenate([[0], np.cumsum(d)])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    part = rng.integers(0, n // 5, n) * 5
    r, r_o = dg.rebuild(part).download(), po.rebuild(g, part)
    assert np.array_equal(r.offs, r_o.offs) and np.array_equal(r.edges.view(np.uint8), r_o.edges.view(np.uint8))
    vdeg, c = po.init_degrees(g)
    st = (np.arange(n), np.ones(n, np.int64), vdeg.copy(), vdeg, c)
    t_o, cw_o, _, _ = po.sweep(g, *st)
    t, cw, _, _ = dg.sweep(*st)
    assert np.array_equal(t, t_o) and np.array_equal(cw.view(np.uint64), cw_o.view(np.uint64))
