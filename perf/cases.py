"""The work that users of this package have it do, as measurable cases.

A case is one call of a public entry point on a graph that the program loaded
once: a batch of BFS, SSSP and WCC queries over it (``Engine.run_batch`` into
device memory, ``Engine.run_batch`` into host memory, the allocation-free
``Engine.run_batch_static``) or a continuous-batching session
(``Engine.serve_*``).  The graph is part of the case (its own seed is in it),
as the data set is part of such a program; the seed given to ``prepare``
makes what changes from call to call, the queries.  Graphs are made here with
torch on the GPU and handed over as CSR arrays.

Every output is a whole number (depths, distances, component labels), laid
out one row of V values per query, -1 where a vertex is not reached (the
library's 0xFFFFFFFF read as int32).
"""
import collections
import ctypes
import math

import numpy as np
import torch

import cgp_amd

# Graph kinds, with the parameters of this repository's benchmark:
#   rmat   R-MAT (0.57 / 0.19 / 0.19 / 0.05), self-loops dropped, symmetrised,
#          deduplicated; V vertices (endpoints past V are dropped), 16 V pairs
#   web    the same without symmetrising: a directed graph, 8 V pairs
#   grid   rows x cols mesh plus 1 % random edges, symmetric (road networks)
# weights: 0 none, else uniform in [1, weights], the same in both directions.
# how: "device" and "host" say where run_batch leaves its results; "static"
# is the allocation-free entry point; "serve" a session of `slots` slots.
_KEYS = ("graph", "v", "cols", "weights", "graph_seed", "bfs", "sssp", "wcc", "how", "slots")


def _case(name, *values):
    c = dict(zip(_KEYS, values))
    return dict({"name": name}, **c) if name else c


def listed():
    return [
        # One interactive lookup on a small graph, the answer in host memory:
        # launches, copies and round trips count.
        _case("rmat12_bfs1_host", "rmat", 1 << 12, 0, 0, 11, 1, 0, 0, "host", 0),
        # A tight loop that may not allocate device memory: a small mixed
        # batch through the static scratch.
        _case("rmat14_mixed20_static", "rmat", 1 << 14, 0, 64, 12, 8, 11, 1, "static", 0),
        # The small batch of the benchmark: 32 BFS at once.
        _case("rmat16_bfs32", "rmat", 1 << 16, 0, 0, 1, 32, 0, 0, "device", 0),
        # One shortest-path query on a mid-sized graph.
        _case("rmat18_sssp1", "rmat", 1 << 18, 0, 64, 13, 0, 1, 0, "device", 0),
        # Directed, odd-sized, borrowed device arrays, a few queries of each kind.
        _case("web300007_mixed21", "web", 300007, 0, 100, 14, 9, 11, 1, "device", 0),
        # A handful of routes on a ragged road network: long, thin frontiers
        # and many iterations.
        _case("grid1001x777_sssp5", "grid", 1001, 777, 1000, 15, 0, 5, 0, "device", 0),
        # Requests served by continuous batching, more of them than slots.
        _case("rmat18_serve40", "rmat", 1 << 18, 0, 64, 13, 28, 12, 0, "serve", 32),
        # Many routes on a large road network.
        _case("grid2048_sssp128", "grid", 2048, 2048, 1000, 5, 0, 128, 0, "device", 0),
        # The benchmark's SSSP batch.
        _case("rmat20_sssp64", "rmat", 1 << 20, 0, 64, 2, 0, 64, 0, "device", 0),
        # The benchmark's headline graph: one query with the components beside
        # it, the BFS share of the batch alone, and the whole mixed batch.
        _case("rmat22_bfs1_wcc1", "rmat", 1 << 22, 0, 255, 3, 1, 0, 1, "device", 0),
        _case("rmat22_bfs160", "rmat", 1 << 22, 0, 255, 3, 160, 0, 0, "device", 0),
        _case("rmat22_mixed256", "rmat", 1 << 22, 0, 255, 3, 160, 80, 16, "device", 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rmat", "rmat", "rmat", "web", "grid"])
    gs = rng.randrange(1, 1000)
    if kind == "grid":
        rows = _log_int(rng, 64, 2048)
        cols = min(2048, int(rows * rng.uniform(0.5, 2.0)))
        n = _log_int(rng, 1, 128)
        bfs = rng.choice([0, 0, n // 2])
        return _case("", kind, rows, cols, rng.choice([100, 1000]), gs, bfs, max(1, n - bfs), rng.randrange(2),
                     "device", 0)
    how = rng.choice(["device", "device", "device", "host", "static", "serve"])
    top = {"device": 1 << 22, "host": 1 << 18, "static": 1 << 16, "serve": 1 << 18}[how]
    v = _log_int(rng, 1 << 12, min(top, 1 << 20) if kind == "web" else top)
    most = {"device": 256, "host": 48, "static": 48, "serve": 48}[how]
    n = _log_int(rng, 1, most)
    mix = rng.choice(["bfs", "sssp", "both", "both"])
    sssp = 0 if mix == "bfs" else max(1, min(80, n if mix == "sssp" else n // 3))
    bfs = 0 if mix == "sssp" else max(1, n - sssp)
    weights = rng.choice([0, 64, 255]) if sssp else rng.choice([0, 64])
    return _case("", kind, v, 0, weights, gs, bfs, sssp, rng.choice([0, 0, 1, 2]), how,
                 rng.choice([16, 32]) if how == "serve" else 0)


def _rand(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(n, generator=g, device="cuda")


def _csr(case):
    """(V, offsets, indices, weights or None) of the case's graph, int32 on the GPU, rows sorted."""
    v, seed = case["v"], case["graph_seed"] * 1000
    if case["graph"] == "grid":
        rows, cols, v = case["v"], case["cols"], case["v"] * case["cols"]
        at = torch.arange(v, device="cuda").view(rows, cols)
        extra = max(1, v // 100)
        a = torch.cat([at[:, :-1].reshape(-1), at[:-1].reshape(-1), (_rand(extra, seed) * v).long().clamp_(max=v - 1)])
        b = torch.cat([at[:, 1:].reshape(-1), at[1:].reshape(-1), (_rand(extra, seed + 1) * v).long().clamp_(max=v - 1)])
    else:
        m = v * (16 if case["graph"] == "rmat" else 8)
        a = torch.zeros(m, dtype=torch.int64, device="cuda")
        b = torch.zeros(m, dtype=torch.int64, device="cuda")
        for bit in range((v - 1).bit_length()):
            r = _rand(m, seed + bit)
            a.mul_(2).add_(r >= 0.76)
            b.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        keep = (a < v) & (b < v)
        a, b = a[keep], b[keep]
    keep = a != b
    a, b = a[keep], b[keep]
    if case["graph"] != "web":
        a, b = torch.cat([a, b]), torch.cat([b, a])
    key = torch.unique(a * v + b)
    del a, b, keep
    src, dst = key // v, key % v
    off = torch.zeros(v + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(src, minlength=v), 0)
    wt = None
    if case["weights"]:
        h = torch.minimum(src, dst) * 1000003 + torch.maximum(src, dst) + seed
        h = ((h ^ (h >> 17)) * 668265263) & 0x7FFFFFFFFFFF
        wt = ((h ^ (h >> 21)) % case["weights"] + 1).int()
    return v, off.int(), dst.int(), wt


class _Array:
    """A torch tensor as the device array that the package's entry points take."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, ctypes.c_void_p(t.data_ptr()), t.numel() * t.element_size()


# The graphs a program has loaded, and its engine on each: (engine, V, source candidates).
_loaded = collections.OrderedDict()


def _load(case):
    spec = tuple(case[k] for k in _KEYS[:5])
    if spec not in _loaded:
        v, off, idx, wt = _csr(case)
        candidates = torch.nonzero(off[1:] > off[:-1]).view(-1).cpu()
        torch.cuda.synchronize()
        if case["graph"] == "web":
            graph = cgp_amd.Graph.from_device(v, idx.numel(), _Array(off), _Array(idx), _Array(wt) if wt is not None else None)
        else:
            graph = cgp_amd.Graph.from_csr(off.cpu().numpy(), idx.cpu().numpy(), wt.cpu().numpy() if wt is not None else None)
        _loaded[spec] = (cgp_amd.Engine(graph), v, candidates)
        while len(_loaded) > 16:
            _loaded.popitem(last=False)[1][0].close()
    _loaded.move_to_end(spec)
    return _loaded[spec]


def prepare(case, seed):
    engine, v, candidates = _load(case)
    g = torch.Generator().manual_seed(seed)
    n = case["bfs"] + case["sssp"]
    sources = candidates[torch.randint(len(candidates), (n,), generator=g)].tolist() + [0] * case["wcc"]
    kinds = [cgp_amd.BFS] * case["bfs"] + [cgp_amd.SSSP] * case["sssp"] + [cgp_amd.WCC] * case["wcc"]
    state = {"engine": engine, "kinds": kinds, "sources": sources, "how": case["how"], "slots": case["slots"]}
    if case["how"] in ("device", "static"):
        state["out"] = _Array(torch.empty((len(kinds), v), dtype=torch.int32, device="cuda"))
    if case["how"] == "serve":  # requests arrive mixed
        order = torch.randperm(len(kinds), generator=g).tolist()
        state["kinds"], state["sources"] = [kinds[i] for i in order], [sources[i] for i in order]
    return state


def run(state):
    engine, kinds, sources = state["engine"], state["kinds"], state["sources"]
    if state["how"] == "device":
        engine.run_batch(kinds, sources, out=state["out"])
        return state["out"].t
    if state["how"] == "static":
        engine.run_batch_static(kinds, sources, state["out"])
        return state["out"].t
    if state["how"] == "host":
        return engine.run_batch(kinds, sources)[0].view(np.int32)
    engine.serve_start(max_slots=state["slots"])
    for i, (kind, source) in enumerate(zip(kinds, sources)):
        engine.serve_submit(kind, source, i, 0.0)
    results = [None] * len(kinds)
    left = len(kinds)
    while left:
        for c in engine.serve_step():
            results[c["ticket"]] = c["result"].view(np.int32)
            left -= 1
    engine.serve_stop()
    return results


def _sizes(case):
    """(V, about E) of the case's graph: duplicates and self-loops of the R-MAT pairs are about a tenth."""
    if case["graph"] == "grid":
        v = case["v"] * case["cols"]
        return v, 4.02 * v
    return case["v"], case["v"] * (28.8 if case["graph"] == "rmat" else 7.2)


def work(case):
    """The graph's arrays read once, every result written once; a comparison
    of every edge for every SSSP query (BFS bits and labels are not counted)."""
    v, e = _sizes(case)
    n = case["bfs"] + case["sssp"] + case["wcc"]
    graph = 4 * (v + 1) + 4 * e + (4 * e if case["weights"] and case["sssp"] else 0)
    return {"bytes": float(graph + 4 * n * v), "flops": float(2 * e * case["sssp"])}


def exact(case, seed):
    """The same rows by plain relaxation of every edge until nothing changes, in 64 bits."""
    v, e = _sizes(case)
    if e * (case["bfs"] + case["sssp"] + min(1, case["wcc"])) > 4e8 or case["graph"] == "grid":
        return None
    v, off, idx, wt = _csr(case)
    candidates = torch.nonzero(off[1:] > off[:-1]).view(-1).cpu()
    src = torch.repeat_interleave(torch.arange(v, device="cuda"), (off[1:] - off[:-1]).long())
    dst, far = idx.long(), 1 << 40
    n = case["bfs"] + case["sssp"]
    g = torch.Generator().manual_seed(seed)
    sources = candidates[torch.randint(len(candidates), (n,), generator=g)].tolist()
    rows = []
    for i in range(n + case["wcc"]):
        if i < n:
            x = torch.full((v,), far, dtype=torch.int64, device="cuda")
            x[sources[i]] = 0
            step = wt.long() if i >= case["bfs"] and wt is not None else 1
        else:  # the smallest vertex of the component, edges taken both ways
            x, step = torch.arange(v, device="cuda"), 0
        while True:
            y = x.scatter_reduce(0, dst, x[src] + step, "amin")
            if i >= n:
                y = y.scatter_reduce(0, src, y[dst], "amin")
            if torch.equal(x, y):
                break
            x = y
        rows.append(torch.where(x >= far, -1, x).int())
    if case["how"] == "serve":
        rows = [rows[i] for i in torch.randperm(len(rows), generator=g).tolist()]
        return [r.cpu().numpy() for r in rows]
    rows = torch.stack(rows)
    return rows.cpu().numpy() if case["how"] == "host" else rows
