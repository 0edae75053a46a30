"""Rebuilds with segments around the sizes where they are split: coarse rows copied in chunks,
overflowing communities emitted in chunks, and runs of fine edges between two communities
folded by a wave.  The coarse CSR equals the oracle's byte for byte, with real weights and with
whole ones."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _graph(deg, run, seed, whole):
    """Vertex 0 with `deg` neighbours; communities A and B of 200 members each, with `run` edges
    between them, and A's members each tied to a vertex of its own (so A overflows)."""
    rng = np.random.default_rng(seed)
    a0, b0, c0 = 1, 201, 401
    n = max(c0 + 200, deg + 1)
    pairs = {(0, v) for v in range(1, deg + 1)}
    pairs |= {(a0 + i, c0 + i) for i in range(200)}
    for k in rng.choice(200 * 200, run, replace=False):
        pairs.add((a0 + int(k) // 200, b0 + int(k) % 200))
    pairs = np.array(sorted(pairs))
    w = rng.integers(1, 50, len(pairs)).astype(float) if whole else rng.uniform(0.1, 1.0, len(pairs))
    cv = np.arange(n)
    cv[a0:a0 + 200] = a0
    cv[b0:b0 + 200] = b0
    return po.from_edge_list(n, pairs, w), cv


@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("deg,run", [(2047, 255), (2048, 256), (2449, 257), (4095, 1023), (4096, 4096), (4097, 4097),
                                     (8192, 8193), (8600, 20000)])
def test_split_segments(ctx, deg, run, whole):
    g, cv = _graph(deg, run, deg + run, whole)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    for part in (cv, np.arange(g.nv), np.where(cv < 401, 0, cv)):
        r, r_o = dg.rebuild(part).download(), po.rebuild(g, part)
        assert np.array_equal(r.offs, r_o.offs)
        assert np.array_equal(r.edges.view(np.uint8), r_o.edges.view(np.uint8))
