"""Batches whose graphs all fit one workgroup, around the sizes where its form changes (2048, 4096
and 8192 vertices, 8193 takes the separate launches): per graph the results of the graph alone,
with hubs and long event runs among the graphs."""
import numpy as np
import pytest

import vite_amd

pytestmark = pytest.mark.gpu


def _graph(ctx, n, i):
    if i % 3 == 2 and n > 40:
        return ctx.gen_ba(n + i, n, 4)
    return ctx.gen_rgg(n + i, n, 1.0 if i % 3 else 0.0)


@pytest.mark.parametrize("largest", [130, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("kw", [dict(), dict(threshold_cycling=True)], ids=["plain", "cycling"])
def test_equals_the_graphs_alone(ctx, largest, kw):
    graphs = [_graph(ctx, n, i) for i, n in enumerate([largest, 65, largest, 100, 1000 % largest + 30, largest])]
    batch = vite_amd.Batch(ctx, graphs)
    for _ in range(2):
        res, stats = batch.run(**kw)
        for g, r in zip(graphs, res):
            o = g.run(**kw)
            assert r.call_q == o.call_q and r.call_iters == o.call_iters
            assert r.level_nv == o.level_nv and r.level_ne == o.level_ne and r.final_q == o.final_q
        calls = max(len(r.call_iters) for r in res)
        assert stats["rounds"] == sum(max(r.call_iters[k] for r in res if len(r.call_iters) > k) for k in range(calls))
    batch.free()
