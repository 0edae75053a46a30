"""Phases on graphs whose degrees are whole numbers: the moves are added to the communities in any
order, with the bits of the oracle's in-order folds; degrees that total 2^52 and more, and a
fraction among them, take the folds in order."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _graph(n, kind):
    """Stars of many sizes (every leaf's best move is its centre) tied together by a path and by
    random edges, with whole weights; `kind` scales them or puts one fraction in."""
    rng = np.random.default_rng(n)
    centre = np.minimum((rng.random(n) ** 4 * 600).astype(np.int64), n - 1)
    pairs = np.concatenate([np.stack([centre, np.arange(n)], 1), np.stack([np.arange(n - 1), np.arange(1, n)], 1),
                            rng.integers(0, n, (n // 2, 2))])
    pairs = np.unique(np.sort(pairs[pairs[:, 0] != pairs[:, 1]], axis=1), axis=0)
    w = np.where((pairs[:, 0] < 600) & (rng.random(len(pairs)) < 0.9), 9.0, 1.0)
    if kind == "large":
        w = w * 2.0 ** 40
    if kind == "fraction":
        w[len(w) // 2] = 0.7
    return po.from_edge_list(n, pairs, w)


@pytest.mark.parametrize("kind", ["whole", "large", "fraction"])
@pytest.mark.parametrize("n", [8193, 9216, 30011])
def test_phases(ctx, n, kind):
    g = _graph(n, kind)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    nc, colors = po.color(g, 4)
    for kw in (dict(), dict(mode="color", num_color=nc + 1, colors=colors), dict(et_type=2, et_delta=0.25),
               dict(mode="vorder", num_color=nc + 1, colors=colors)):
        q_o, cv_o, it_o = po.louvain_phase(g, **kw)
        q, cv, it = dg.louvain_phase(sequential=True, **kw)
        assert (q, it) == (q_o, it_o) and np.array_equal(cv, cv_o), kw
    st = dg.phase_begin(thresh=-1.0)
    for _ in range(3):
        st.step()
    s = st.state()
    st.end(want_cvect=False)
    if kind == "whole":  # the community state after three rounds of moves
        assert np.array_equal(s["cdeg"], np.bincount(s["curr"], s["vdeg"], n))
        assert np.array_equal(s["csize"], np.bincount(s["curr"], minlength=n))
