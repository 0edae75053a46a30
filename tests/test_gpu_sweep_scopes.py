"""What a sweep's launches are timed as: one "local_move_hub" around all the work on hub rows, however many
launches it takes, and the launch of buckets 0 to 3 together under a name of its own."""
import numpy as np
import pytest

import bench
import vite_amd
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _counts(ctx, dg, names):
    st = dg.phase_begin(thresh=-1.0)
    ctx.set_profiling(True)
    ctx.reset_stats()
    st.sweep()
    n = {k: ctx.kernel_stats(k)[1] for k in names}
    ctx.set_profiling(False)
    st.end(want_cvect=False)
    return n


@pytest.mark.parametrize("long,whole,expect", [([], False, dict(hub_lds=3)), ([5000] * 3, True, dict(hub_lds=3, hubw_insert=1)),
                                               ([5000] * 3, False, dict(hub_own=1))])
def test_hub_rows_are_one_scope(ctx, long, whole, expect):
    n, rng = 9000, np.random.default_rng(len(long))
    d = rng.integers(0, 6, n)
    d[:300] = 600
    d[:6] = [1024, 1025, 2048, 2049, 3000, 4096]
    d[300:300 + len(long)] = long
    offs = np.concatenate([[0], np.cumsum(d)])
    w = rng.integers(1, 9, offs[-1]).astype(float) if whole else rng.uniform(0.1, 1.0, offs[-1])
    g = po.make_graph(offs, rng.integers(0, n, offs[-1]), w)
    dg = ctx.upload(vite_amd.CSR(g.offs, g.edges))
    n_of = _counts(ctx, dg, ["local_move_hub", "hub_lds", "hubw_insert", "hub_own"])
    assert n_of == {**dict(local_move_hub=1, hub_lds=0, hubw_insert=0, hub_own=0), **expect}


def test_one_launch_of_a_small_graph(ctx):
    names = ["local_move", "local_move_rest", "local_move_all"]
    assert _counts(ctx, ctx.gen_rgg(3, 20000, 1.0), names) == dict(local_move=0, local_move_rest=0, local_move_all=1)
    assert _counts(ctx, ctx.gen_rgg(3, 1 << 19, 1.0), names) == dict(local_move=1, local_move_rest=1, local_move_all=0)
    assert bench.g16_kernel({}) == "k_local_move<false, 2, false>"
    assert bench.g16_kernel({}, True) == "k_local_move<false, 3, false>"
