"""The work this framework is measured on: whole community-detection jobs through the public
Python entry points, from a thousand vertices to half a billion directed entries.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the graphs and handles a program holds before the call
    run(state)           one pass
    work(case)           bytes and operations of one pass that cannot be done without
    exact(case, seed)    the same results from plain numpy in 64 bits

Graphs are random geometric (radius sqrt(2 ln n / (pi n)), weights the distances, optionally 1%
further edges of weight U(0,1)) or Barabasi-Albert with m attachments, as in bench.py and
tests/.  "own" graphs are built by the caller on the host and uploaded, the others come from
the device generators.
"""
import math

import numpy as np

import vite_amd

_ctx = None


def _context():
    """One context for the program, as a user's process holds it."""
    global _ctx
    if _ctx is None:
        _ctx = vite_amd.Context(0)
    return _ctx


def _run_case(name, graph, n, **more):
    c = dict(name=name, kind="run", graph=graph, n=n, extra=0.0, m=0, cycling=False, coloring=False,
             vertex_order=False, et=0, delta=1.0)
    c.update(more)
    return c


def listed():
    return [
        # a caller's own small graph: uploaded, clustered, freed (launches and host time count)
        _run_case("job_rgg_1k", "own", 1000, kind="job"),
        # the benchmark's small configuration: RGG n = 65536 at threshold 1e-6
        _run_case("run_rgg_64k", "own", 65536),
        # a serving-size skewed graph, not a power of two, with threshold cycling (-i)
        _run_case("run_ba_300k", "ba", 300007, m=8, cycling=True),
        # the largest serving size: RGG n = 2^20 with 1% extra edges, -i
        _run_case("run_rgg_1m", "rgg", 1 << 20, extra=1.0, cycling=True),
        # the headline graph: RGG n = 2^24 with 1% extra edges (563 M entries), -i
        _run_case("run_rgg_16m", "rgg", 1 << 24, extra=1.0, cycling=True),
        # the skewed configuration: BA n = 2^22, m = 8, -c 8 -t 2 -a 0.25
        _run_case("run_ba_4m_color_et", "ba", 1 << 22, m=8, coloring=True, et=2, delta=0.25),
        # vertex ordering with early termination (-d 8 -t 1) on an ordinary odd size
        _run_case("run_rgg_777k_order_et", "rgg", 777001, extra=1.0, vertex_order=True, et=1),
        # one level by hand, as a caller of the phase and rebuild entry points drives it
        dict(name="level_rgg_4m", kind="level", graph="rgg", n=4200001, extra=1.0, m=0),
        # a few hundred small graphs in one call
        dict(name="batch_300_small", kind="batch", count=300, lo=256, hi=4096),
        # the batched configuration: 4096 RGGs, n log-uniform in [2^8, 2^16], 1% extra on half
        dict(name="batch_4096", kind="batch", count=4096, lo=256, hi=65536),
        # a burst of requests to the serving loop: RGG and BA (m = 8) in turn
        dict(name="serve_48", kind="serve", count=48, lo=1024, hi=262144),
        # a partition against its ground truth (-g)
        dict(name="compare_1m", kind="compare", n=1000003, groups=30011),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["job", "run", "run", "run", "run", "level", "batch", "compare"])
    if kind == "job":
        return {k: v for k, v in _run_case("", "own", _log_int(rng, 300, 20000), kind="job",
                                           cycling=rng.random() < 0.5).items() if k != "name"}
    if kind == "run":
        ba = rng.random() < 0.4
        c = _run_case("", "ba" if ba else "rgg", _log_int(rng, 1024, 1 << 20 if ba else 1 << 23),
                      m=rng.choice([4, 8]) if ba else 0, extra=0.0 if ba else rng.choice([0.0, 1.0]))
        form = rng.choice(["plain", "cycling", "cycling", "color", "order"])
        c["cycling"] = form == "cycling"
        c["coloring"] = form == "color"
        c["vertex_order"] = form == "order"
        if form in ("color", "order"):
            c["et"] = rng.choice([0, 1, 2])
            c["delta"] = 0.25
        del c["name"]
        return c
    if kind == "level":
        return dict(kind="level", graph="rgg", n=_log_int(rng, 1 << 15, 1 << 22), extra=rng.choice([0.0, 1.0]), m=0)
    if kind == "batch":
        lo = _log_int(rng, 128, 2048)
        return dict(kind="batch", count=_log_int(rng, 32, 1024), lo=lo, hi=_log_int(rng, 2 * lo, 65536))
    n = _log_int(rng, 3000, 4000000)
    return dict(kind="compare", n=n, groups=_log_int(rng, 2, max(3, n // 8)))


# ---- inputs ---------------------------------------------------------------------------------

def _sizes(case):
    """Vertex counts of a batch or burst: the quantiles of the log-uniform law on [lo, hi], in
    an order without trend."""
    k, lo, hi = case["count"], case["lo"], case["hi"]
    q = (np.arange(k) + 0.5) / k
    n = np.rint(np.exp(math.log(lo) + q * (math.log(hi) - math.log(lo)))).astype(np.int64)
    return [int(x) for x in n[np.argsort((np.arange(k) * 0.6180339887498949) % 1.0)]]


def _geometric(seed, n):
    """A random geometric graph on the host: (offsets, tails, weights), vertices numbered cell by
    cell, rows ascending."""
    r = math.sqrt(2.0 * math.log(n) / (math.pi * n))
    nc = max(1, int(1.0 / r))
    p = np.random.default_rng(seed).random((n, 2))
    cell = np.minimum((p[:, 1] * nc).astype(np.int64), nc - 1) * nc + np.minimum((p[:, 0] * nc).astype(np.int64), nc - 1)
    order = np.argsort(cell, kind="stable")
    p, cell = p[order], cell[order]
    start = np.searchsorted(cell, np.arange(nc * nc + 1))
    x, y = p[:, 0].copy(), p[:, 1].copy()
    cx, cy = cell % nc, cell // nc
    src, dst = [], []
    for oy in (-1, 0, 1):
        # the three cells of one row of the neighbourhood hold consecutive vertices
        yy = cy + oy
        ok = np.flatnonzero((yy >= 0) & (yy < nc))
        a = start[yy[ok] * nc + np.maximum(cx[ok] - 1, 0)]
        b = start[yy[ok] * nc + np.minimum(cx[ok] + 1, nc - 1) + 1]
        cnt = b - a
        s = np.repeat(ok, cnt)
        t = np.arange(cnt.sum()) - np.repeat(np.cumsum(cnt) - cnt, cnt) + np.repeat(a, cnt)
        near = ((x[s] - x[t]) ** 2 + (y[s] - y[t]) ** 2 <= r * r) & (s != t)
        src.append(s[near])
        dst.append(t[near])
    s, t = np.concatenate(src), np.concatenate(dst)
    o = np.argsort(s * n + t)
    s, t = s[o], t[o]
    offs = np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))])
    return offs, t, np.sqrt((x[s] - x[t]) ** 2 + (y[s] - y[t]) ** 2)


def _device_graph(case, seed):
    ctx = _context()
    if case["graph"] == "own":
        return ctx.upload(vite_amd.CSR.from_arrays(*_geometric(seed, case["n"])))
    if case["graph"] == "ba":
        return ctx.gen_ba(seed, case["n"], case["m"])
    return ctx.gen_rgg(seed, case["n"], case["extra"])


def _partitions(case, seed):
    """Two labelings of the same vertices: a truth of uneven groups and a found partition that
    agrees with it on most vertices."""
    rng = np.random.default_rng(seed)
    n, k = case["n"], case["groups"]
    truth = np.minimum((k * rng.random(n) ** 1.5).astype(np.int64), k - 1)
    found = np.where(rng.random(n) < 0.15, rng.integers(0, k, n), truth)
    return truth, found


def prepare(case, seed):
    kind = case["kind"]
    if kind == "job":
        return dict(case=case, csr=vite_amd.CSR.from_arrays(*_geometric(seed, case["n"])))
    if kind in ("run", "level"):
        return dict(case=case, g=_device_graph(case, seed))
    if kind == "batch":
        ctx = _context()
        graphs = [ctx.gen_rgg(seed * 100003 + i, n, 1.0 if i % 2 else 0.0) for i, n in enumerate(_sizes(case))]
        batch = vite_amd.Batch(ctx, graphs)
        for g in graphs:
            g.free()
        return dict(case=case, batch=batch)
    if kind == "serve":
        return dict(case=case, server=vite_amd.Server(hbm_budget=64 << 30, slots=4), seed=seed, sizes=_sizes(case))
    truth, found = _partitions(case, seed)
    return dict(case=case, truth=truth, found=found)


# ---- one pass -------------------------------------------------------------------------------

def _options(case):
    return dict(threshold_cycling=case["cycling"], coloring=case["coloring"], vertex_order=case["vertex_order"],
                et_type=case["et"], et_delta=case["delta"])


def _padded(values, length, dtype):
    """Lists whose length depends on the run, in arrays that always have the same shape."""
    out = np.full(length, -1, dtype)
    out[: len(values)] = values
    return out


def _result(r):
    return dict(final_q=np.array(r.final_q), call_q=_padded(r.call_q, 32, float), call_iters=_padded(r.call_iters, 32, np.int64),
                level_q=_padded(r.level_q, 32, float), level_iters=_padded(r.level_iters, 32, np.int64),
                level_nv=_padded(r.level_nv, 32, np.int64), level_ne=_padded(r.level_ne, 32, np.int64),
                total_iters=r.total_iters, num_colors=r.num_colors)


def _results(rs):
    """Many results as a few arrays."""
    k = 32 * len(rs)
    return dict(final_q=np.array([r.final_q for r in rs]), total_iters=np.array([r.total_iters for r in rs]),
                call_q=_padded([q for r in rs for q in r.call_q], k, float),
                call_iters=_padded([i for r in rs for i in r.call_iters], k, np.int64),
                level_nv=_padded([i for r in rs for i in r.level_nv], k, np.int64),
                level_ne=_padded([i for r in rs for i in r.level_ne], k, np.int64))


def _numbers(stats):
    return {k: np.array(v) for k, v in stats.items()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "job":
        g = _context().upload(state["csr"])
        out = _result(g.run(**_options(case)))
        g.free()
        return out
    if kind == "run":
        return _result(state["g"].run(**_options(case)))
    if kind == "level":
        g = state["g"]
        q0, _, it0 = g.louvain_phase(thresh=1e-3, want_cvect=False)
        trace_q, trace_moves = g.last_trace()
        coarse = g.rebuild()
        q1, cvect, it1 = coarse.louvain_phase(thresh=1e-3)
        out = dict(q=np.array([q0, q1]), iters=np.array([it0, it1]), trace_q=_padded(trace_q, 256, float),
                   trace_moves=_padded(trace_moves, 256, np.int64), nv=coarse.nv, ne=coarse.ne,
                   cvect=np.zeros(case["n"], np.int64))
        out["cvect"][: len(cvect)] = cvect  # the coarse graph's partition, about n / 8 vertices
        coarse.free()
        return out
    if kind == "batch":
        rs, _ = state["batch"].run(threshold_cycling=True)
        return _results(rs)
    if kind == "serve":
        s = state["server"]
        tickets = [s.submit("rgg" if i % 2 else "ba", state["seed"] * 1009 + i, n, 0.0 if i % 2 else 8,
                            threshold_cycling=True) for i, n in enumerate(state["sizes"])]
        return _results([s.wait(t)[0] for t in tickets])
    return _numbers(_context().compare_communities(state["truth"], state["found"]))


# ---- what a pass cannot do without ----------------------------------------------------------

def _csr_bytes(graph, n, extra, m):
    """The CSR's expected bytes: 16 per directed entry, 8 per row start."""
    if graph == "ba":
        e = 2.0 * n * m
    else:
        e = 2.0 * n * math.log(n) * (1.0 + extra / 100.0)
    return 16.0 * e + 8.0 * (n + 1)


def work(case):
    kind = case["kind"]
    if kind == "compare":
        return dict(bytes=16.0 * case["n"], flops=0.0)
    if kind == "batch":
        b = sum(_csr_bytes("rgg", n, 1.0 if i % 2 else 0.0, 0) for i, n in enumerate(_sizes(case)))
    elif kind == "serve":  # the graphs are written by the generators and read
        b = 2.0 * sum(_csr_bytes("rgg" if i % 2 else "ba", n, 0.0, 8) for i, n in enumerate(_sizes(case)))
    else:
        b = _csr_bytes(case["graph"], case["n"], case["extra"], case["m"])
    # two additions per entry (its community's weight, the vertex degree)
    return dict(bytes=b, flops=2.0 * b / 16.0)


# ---- the same results in plain numpy --------------------------------------------------------

def _phase(offs, tail, w, thresh, lower=-1.0):
    """One plain Louvain phase in 64 bits: (modularity, partition, iterations)."""
    n = len(offs) - 1
    src = np.repeat(np.arange(n), np.diff(offs))
    deg = np.bincount(src, w, n)
    c = 1.0 / deg.sum()
    loops = tail == src
    self_w = np.bincount(src[loops], w[loops], n)
    past, curr = np.arange(n), np.arange(n)
    cdeg, csize = deg.copy(), np.ones(n, np.int64)
    prev, iters = lower, 0
    while True:
        iters += 1
        key, inv = np.unique(src * n + curr[tail], return_inverse=True)
        e = np.bincount(inv, w, len(key))
        v, comm = key // n, key % n
        own = comm == curr[v]
        ecc = np.zeros(n)
        ecc[v[own]] = e[own]
        gain = 2.0 * (e - (ecc - self_w)[v]) - 2.0 * deg[v] * (cdeg[comm] - (cdeg[curr] - deg)[v]) * c
        gain[own | ~(gain > 0.0)] = 0.0
        best = np.zeros(n)
        np.maximum.at(best, v, gain)
        pick = np.flatnonzero((gain > 0.0) & (gain == best[v]))[::-1]  # the smallest id is written last
        target = curr.copy()
        target[v[pick]] = comm[pick]
        target = np.where((csize[target] == 1) & (csize[curr] == 1) & (target > curr), curr, target)
        mv = np.flatnonzero(target != curr)
        ids = np.stack([target[mv], curr[mv]], 1).ravel()
        cdeg = cdeg + np.bincount(ids, np.stack([deg[mv], -deg[mv]], 1).ravel(), n)
        csize = csize + np.bincount(target[mv], minlength=n) - np.bincount(curr[mv], minlength=n)
        q = abs(ecc.sum() * c - np.square(cdeg).sum() * c * c)
        if q - prev < thresh:
            return prev, past, iters
        prev = max(q, lower)
        past, curr = curr, target


def _coarse(offs, tail, w, part):
    """The next level: communities numbered by first appearance."""
    n = len(offs) - 1
    _, first, inv = np.unique(part, return_index=True, return_inverse=True)
    rank = np.empty(len(first), np.int64)
    rank[np.argsort(first)] = np.arange(len(first))
    new, nc = rank[inv], len(first)
    src = np.repeat(np.arange(n), np.diff(offs))
    key, kinv = np.unique(new[src] * nc + new[tail], return_inverse=True)
    ne = np.concatenate([[0], np.cumsum(np.bincount(key // nc, minlength=nc))])
    return ne, key % nc, np.bincount(kinv, w, len(key))


def _louvain(offs, tail, w, cycling):
    """The phase loop (plain Louvain, threshold 1e-6 or threshold cycling)."""
    out = dict(call_q=[], call_iters=[], level_q=[], level_iters=[], level_nv=[], level_ne=[])
    prev, total, phase = -1.0, 0, 0

    def call(thresh, lower=-1.0):
        q, part, iters = _phase(offs, tail, w, thresh, lower)
        out["call_q"].append(q)
        out["call_iters"].append(iters)
        return q, part, iters

    while True:
        short = phase % 13
        thresh = (1e-3 if short <= 2 else 1e-4 if short <= 6 else 1e-5 if short <= 9 else 1e-6) if cycling else 1e-6
        nv, ne = len(offs) - 1, len(tail)
        q, part, iters = call(thresh)
        total += iters
        if not q - prev > thresh:
            if cycling and phase < 10:
                q, _, _ = call(1e-6, q)  # the last pass starts from this modularity
            break
        offs, tail, w = _coarse(offs, tail, w, part)
        out["level_q"].append(q)
        out["level_iters"].append(total)
        out["level_nv"].append(nv)
        out["level_ne"].append(ne)
        prev = q
        phase += 1
    out = {k: _padded(v, 32, float if k.endswith("_q") else np.int64) for k, v in out.items()}
    return dict(out, final_q=np.array(q), total_iters=total, num_colors=0)


def _gini(size):
    s = np.sort(size).astype(np.int64)
    k = len(s)
    return (2.0 * float(((np.arange(k) + 1) * s).sum())) / (k * float(s.sum())) - (k + 1.0) / k


def exact(case, seed):
    if case["kind"] == "compare":
        truth, found = _partitions(case, seed)
        size = lambda x: np.bincount(x)  # noqa: E731
        pairs = lambda k: int((k * (k - 1) // 2).sum())  # noqa: E731
        both = np.unique(truth * (int(found.max()) + 1) + found, return_counts=True)[1]
        ss = pairs(both)
        sd, ds = pairs(size(truth)) - ss, pairs(size(found)) - ss
        prec, rec = ss / (ss + ds), ss / (ss + sd)
        return _numbers(dict(n=case["n"], nc_truth=int(truth.max()) + 1, nc_found=int(found.max()) + 1, same_same=ss,
                             same_diff=sd, diff_same=ds, precision=prec, recall=rec,
                             f_score=2.0 * (prec * rec / (prec + rec)), gini_truth=_gini(size(truth)),
                             gini_found=_gini(size(found))))
    # the other kinds' graphs come from the device generators, or take minutes in numpy
    if case["kind"] not in ("job", "run") or case["graph"] != "own":
        return None
    return _louvain(*_geometric(seed, case["n"]), case["cycling"])
