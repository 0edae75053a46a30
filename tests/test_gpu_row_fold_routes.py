"""Vertex degrees of graphs with many long rows: the oracle's bits, and real weights take no multiple of the
time of whole ones where a workgroup's rows are folded by its waves side by side."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _graph(deg, kind, seed):
    rng = np.random.default_rng(seed)
    offs = np.concatenate([[0], np.cumsum(deg)])
    w = rng.uniform(0.1, 1.0, offs[-1])
    if kind != "real":
        w = rng.integers(1, 9, offs[-1]).astype(float)
    if kind == "late":  # every third row ends with a fraction
        w[offs[1::3] - 1] += 0.25
    if kind == "early":  # or begins with one
        w[offs[:-1:3]] += 0.25
    return po.make_graph(offs, rng.integers(0, len(deg), offs[-1]), w)


def _degrees(rows):
    rng = np.random.default_rng(7)
    few = rng.integers(0, 5, 9000)  # a handful of long rows among short ones, two in a workgroup's stretch
    few[rng.choice(9000, 40, replace=False)] = rng.choice([511, 512, 2047, 2048, 4096, 4097, 4160, 9000], 40)
    many = rng.integers(4000, 4300, 700)
    wide = np.where(rng.random(66000) < 0.04, rng.choice([513, 2047, 2048, 2500, 4097], 66000), 20)
    return {"few": few, "many": many, "wide": wide}[rows]


@pytest.mark.parametrize("kind", ["real", "whole", "late", "early"])
@pytest.mark.parametrize("rows", ["few", "many", "wide"])
def test_degrees(ctx, rows, kind):
    g = _graph(_degrees(rows), kind, 5)
    vdeg, c = po.init_degrees(g)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    v, _ = dg.init_degrees()
    assert np.array_equal(v.view(np.uint64), vdeg.view(np.uint64))
    _, c_seq = dg.init_degrees(sequential=True)
    assert c_seq == c
    # the phase's state, and the route of its moves, come from the same degrees
    q_o, cv_o, it_o = po.louvain_phase(g, thresh=1e-2)
    q, cv, it = dg.louvain_phase(sequential=True, thresh=1e-2)
    assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o)


def test_time_of_long_real_rows(ctx):
    best = {}
    for kind in ("real", "whole"):
        rng = np.random.default_rng(1)
        g = _graph(rng.integers(5000, 6000, 4000), kind, 3)
        dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
        for _ in range(5):
            ctx.set_profiling(True)
            ctx.reset_stats()
            dg.init_degrees()
            best[kind] = min(best.get(kind, np.inf), ctx.kernel_stats("row_fold")[2])
            ctx.set_profiling(False)
    # 2.3 with a wave per row; one wave of a workgroup folding all of its rows took 5.4 times as long
    assert 0 < best["real"] < 4 * best["whole"], best
