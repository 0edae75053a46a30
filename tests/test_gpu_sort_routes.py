"""The vertex sorts' two forms: the library's for few pairs, the device sort's launches where they are fewer.
A generated graph's points, a rebuild's members and a sweep's lists around the lines between them
equal the oracle's."""
import numpy as np
import pytest

import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,parts,device", [(1000, 0, False), (4096, 0, False), (30000, 0, False), (9000, 200, True),
                                            (65536, 60000, False), (65537, 60000, True), (131073, 100000, True)])
def test_routes(ctx, n, parts, device):
    """A generated graph sorts its points by cell (more than 8 bits from a few thousand points on); a
    rebuild sorts the vertices by community."""
    if parts == 0:
        launch = lambda: ctx.gen_rgg(n, n, 1.0).free()  # noqa: E731
    else:
        rng = np.random.default_rng(n)
        d = rng.integers(0, 4, n)
        offs = np.concatenate([[0], np.cumsum(d)])
        g = po.make_graph(offs, rng.integers(0, n, offs[-1]), rng.uniform(0.1, 1.0, offs[-1]))
        dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
        part = rng.permutation(np.concatenate([np.arange(parts), rng.integers(0, parts, n - parts)]))
        r, r_o = dg.rebuild(part).download(), po.rebuild(g, part)
        assert np.array_equal(r.offs, r_o.offs) and np.array_equal(r.edges.view(np.uint8), r_o.edges.view(np.uint8))
        launch = lambda: dg.rebuild(part).free()  # noqa: E731
    ctx.set_profiling(True)
    ctx.reset_stats()
    launch()
    sorts, passes = ctx.kernel_stats("sort_u32")[1], ctx.kernel_stats("dsort_scatter")[1]
    ctx.set_profiling(False)
    assert sorts == (0 if device else 1) and (passes > 0) == device
