"""Near-far postponing of SSSP pairs where a run is cut, served, or shares its
iterations with other queries.  Every row is compared with the oracle or with
distances that follow from the graph's shape."""
import numpy as np
import pytest

import cgp_amd
import oracle_lib as O
from cgp_amd import BFS, SSSP

pytestmark = pytest.mark.gpu
INF = 0xFFFFFFFF


def csr(V, src, dst, wt):
    """CSR arrays of the edges, rows sorted."""
    order = np.lexsort((dst, src))
    off = np.zeros(V + 1, np.int64)
    np.add.at(off, np.asarray(src) + 1, 1)
    return (np.cumsum(off).astype(np.int32), np.asarray(dst)[order].astype(np.int32),
            np.asarray(wt)[order].astype(np.uint32))


def path(V, w):
    a = np.arange(V - 1)
    return csr(V, np.concatenate([a, a + 1]), np.concatenate([a + 1, a]), np.full(2 * V - 2, w))


# A path of V vertices of weight 90 from its first vertex: each counted iteration
# settles one more hop, however many raises of the threshold lie between (one
# per hop at steps up to 90, one per 20 hops at the automatic 20 x 90).
@pytest.mark.parametrize("delta", [0, 30, 200, -1])
@pytest.mark.parametrize("kinds", [[SSSP], [SSSP] * 5 + [BFS] * 3, [BFS] * 70 + [SSSP] * 9])
@pytest.mark.parametrize("opts", [dict(), dict(frontier_dense_div=1, dense_threshold=1), dict(use_hip_graph=0)],
                         ids=["default", "rows", "direct"])
def test_iteration_limit(gpu, delta, kinds, opts):
    V = 300
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(*path(V, 90)), sssp_delta=delta, **opts)
    hops = np.arange(V, dtype=np.uint32)
    out = cgp_amd.DeviceBuffer(len(kinds) * V * 4)
    for k in (1, 2, 21, 45, V - 2, V - 1, V):
        en.set_opts(max_iterations=k)
        got = en.run_batch(kinds, [0] * len(kinds))[0]
        en.run_batch_static(kinds, [0] * len(kinds), out)
        for i, kind in enumerate(kinds):
            exp = np.where(hops <= k, hops * (90 if kind == SSSP else 1), INF).astype(np.uint32)
            assert np.array_equal(got[i], exp), (k, i, kind)
            assert np.array_equal(out.to_host(shape=(len(kinds), V))[i], exp), (k, i, kind, "static")


def serve(en, queries, slots, max_iterations=1):
    """Completions by ticket of a session that has all queries from the start."""
    en.serve_start(max_slots=slots)
    for i, (kind, source) in enumerate(queries):
        en.serve_submit(kind, source, i, 0.0)
    done = {}
    while len(done) < len(queries):
        for c in en.serve_step(max_iterations=max_iterations):
            done[c["ticket"]] = c
    en.serve_stop()
    return done


# Two parts: 0 -> 2 at 100 and 0 -> 1 -> 2 at 10 each (vertex 2 is put into the
# far set at 100 and then lowered below the threshold of 50, which leaves its
# bit there), and a path of weight 1 whose queries stay below the threshold.  The
# queries of the first part are done after their third or fourth iteration,
# whoever else is running, and their slot serves the next one.
@pytest.mark.parametrize("first", [SSSP, BFS])
@pytest.mark.parametrize("slots", [2, 64, 128])
def test_completion_beside_others(gpu, slots, first):
    n = 45
    a = np.arange(3, 3 + n)
    off, idx, wt = csr(4 + n, np.concatenate([[0, 0, 1], a]), np.concatenate([[2, 1, 2], a + 1]),
                       np.concatenate([[100, 10, 10], np.ones(n)]))
    og = O.G(off, idx, wt)
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt), sssp_delta=50)
    queries = [(SSSP, 3), (SSSP, 0)] + [(first if i % 2 else SSSP, 0) for i in range(5)]
    done = serve(en, queries, slots)
    for i, (kind, source) in enumerate(queries):
        assert np.array_equal(done[i]["result"], O.expected(og, kind, source)), i
        if source == 0:
            assert done[i]["iterations"] <= 4, (i, done[i]["iterations"])
    assert done[0]["iterations"] >= n


# Sessions of one to eight mask words on a road network: queries of every word
# wait at the threshold while others run.
@pytest.mark.parametrize("slots", [16, 128, 300, 512])
@pytest.mark.parametrize("delta", [300, -1])
def test_serving_mask_words(gpu, slots, delta):
    h = cgp_amd.HostCSR.grid(37, 41, p_extra=0.01, seed=7, wmin=1, wmax=1000)
    og = O.G.of(h)
    en = cgp_amd.Engine(cgp_amd.Graph.from_host(h), sssp_delta=delta)
    assert en.opts["sssp_delta"] > 0
    src = h.sample_sources(min(h.V, slots + slots // 2), seed=slots)
    queries = [(SSSP if i % 4 else BFS, int(s)) for i, s in enumerate(src)]
    done = serve(en, queries, slots, max_iterations=0 if slots == 300 else 2)
    for i, (kind, source) in enumerate(queries):
        assert np.array_equal(done[i]["result"], O.expected(og, kind, source)), (i, kind, source)


# The automatic step: road networks have it, also with a vertex of many
# neighbours (here 130 of 16 700 edges); graphs with more of their edges at such
# vertices (1600 of 19 700, or a power law) do not.  Graphs from host and device
# arrays agree.
@pytest.mark.parametrize("graph,on", [("grid", True), ("hub", True), ("hubs", False), ("web", False)])
def test_automatic_step(gpu, graph, on):
    if graph == "web":
        V, rng = 5000, np.random.RandomState(3)
        key = np.unique((V * rng.rand(7 * V) ** 4).astype(np.int64) * V + rng.randint(0, V, 7 * V))
        src, dst = key // V, key % V
        wt = rng.randint(1, 101, len(src))
    else:
        h = cgp_amd.HostCSR.grid(64, 64, p_extra=0.01, seed=3, wmin=1, wmax=100)
        V, rng = h.V, np.random.RandomState(1)
        src, dst, wt = np.repeat(np.arange(V), np.diff(h.offsets)), h.indices, h.weights
        for hub, degree in ([(2000, 130)] if graph == "hub" else [(7, 800), (2000, 800)] if graph == "hubs" else []):
            leaves = rng.choice(np.arange(2001, V), degree, replace=False)
            src = np.concatenate([src, leaves, np.full(degree, hub)])
            dst = np.concatenate([dst, np.full(degree, hub), leaves])
            wt = np.concatenate([wt, np.arange(2 * degree) % degree % 100 + 1])
    off, idx, w = csr(V, src, dst, wt)
    assert len(idx) / V <= 8
    og = O.G(off, idx, w)
    bufs = [cgp_amd.DeviceBuffer.from_array(x) for x in (off, idx, w)]
    for g in (cgp_amd.Graph.from_csr(off, idx, w), cgp_amd.Graph.from_device(V, len(idx), *bufs)):
        en = cgp_amd.Engine(g)
        assert en.opts["sssp_delta"] == (int(round(20 * w.mean(dtype=np.float64))) if on else 0)
        sources = [0, 2000, V - 1, 7, 5]
        got = en.run_batch([SSSP] * 5, sources)[0]
        for i, s in enumerate(sources):
            assert np.array_equal(got[i], O.expected(og, SSSP, s)), (i, s)


# Allocation-free runs: the far words lie behind the records in the fixed array.
# Wide and narrow batches in turn on one engine, several passes, an odd number of
# vertices.
@pytest.mark.parametrize("V", [63, 1501, 5001])
@pytest.mark.parametrize("opts", [dict(), dict(max_words=1), dict(frontier_dense_div=1, dense_threshold=1)],
                         ids=["default", "passes", "rows"])
def test_static_runs(gpu, V, opts):
    rng = np.random.RandomState(V)
    a, b = np.arange(V), np.roll(np.arange(V), -1)
    a, b = np.concatenate([a, rng.randint(0, V, V)]), np.concatenate([b, rng.randint(0, V, V)])
    w = rng.randint(1, 98, len(a))
    off, idx, wt = csr(V, np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w]))
    og = O.G(off, idx, wt)
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt), sssp_delta=60, **opts)
    out = cgp_amd.DeviceBuffer(150 * V * 4)
    for n in (150, 3, 70, 1, 150):
        kinds = [SSSP if i % 3 else BFS for i in range(n)]
        src = [(i * 31 + n) % V for i in range(n)]
        en.run_batch_static(kinds, src, out)
        got = out.to_host(shape=(150, V))
        for i, (k, s) in enumerate(zip(kinds, src)):
            assert np.array_equal(got[i], O.expected(og, k, s)), (n, i, k, s)


# The push launch, which takes up the far set, on a second stream beside the
# lane-per-query launch; captured, launched directly, and in a session.
@pytest.mark.parametrize("n", [5, 40, 150])
@pytest.mark.parametrize("opts", [dict(), dict(use_hip_graph=0), dict(dense_threshold=1)],
                         ids=["graph", "direct", "rows"])
def test_concurrent_advance(gpu, n, opts):
    h = cgp_amd.HostCSR.grid(45, 51, p_extra=0.01, seed=9, wmin=1, wmax=1000)
    og = O.G.of(h)
    en = cgp_amd.Engine(cgp_amd.Graph.from_host(h), sssp_delta=700, concurrent_advance=1, **opts)
    src = [int(s) for s in h.sample_sources(n, seed=n)]
    queries = [(BFS if i % 5 == 4 else SSSP, s) for i, s in enumerate(src)]
    exp = [O.expected(og, k, s) for k, s in queries]
    for _ in range(2):
        got = en.run_batch([k for k, _ in queries], src)[0]
        assert np.array_equal(got, np.stack(exp))
    done = serve(en, queries, 64)
    for i in range(n):
        assert np.array_equal(done[i]["result"], exp[i]), i
