"""GPU parity at the sizes where a launch changes shape: the edges of a
workgroup's share of vertices, edges and work items, and lists shorter and
longer than the launch has waves.  Every row is compared with the oracle."""
import numpy as np
import pytest

import cgp_amd
import oracle_lib as O
from cgp_amd import BFS, SSSP, WCC

pytestmark = pytest.mark.gpu


def ring_graph(V, hub_degree=0, seed=1, chords=3, directed=False):
    """A ring of V vertices with random chords; vertex V // 2 is joined to
    hub_degree others."""
    rng = np.random.RandomState(seed)
    a, b = [np.arange(V)], [(np.arange(V) + 1) % max(V, 1)]
    if V > 4:
        a.append(rng.randint(0, V, chords * V))
        b.append(rng.randint(0, V, chords * V))
    if hub_degree:
        a.append(np.full(hub_degree, V // 2))
        b.append(rng.choice(V, hub_degree, replace=False))
    a, b = np.concatenate(a), np.concatenate(b)
    a, b = a[a != b], b[a != b]
    if not directed:
        a, b = np.concatenate([a, b]), np.concatenate([b, a])
    key = np.unique(a.astype(np.int64) * V + b)
    src, dst = key // V, key % V
    lo, hi = np.minimum(src, dst), np.maximum(src, dst)
    wt = ((lo * 7919 + hi * 104729 + seed) % 97 + 1).astype(np.uint32)
    off = np.zeros(V + 1, np.int64)
    np.add.at(off, src + 1, 1)
    return np.cumsum(off).astype(np.int32), dst.astype(np.int32), wt


def check(off, idx, wt, kinds, sources, runs=1, **opts):
    """Batches of the queries, the sources rotated from run to run on one
    engine (so captured launches are replayed), against the oracle."""
    V = len(off) - 1
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt), **opts)
    og = O.G(off, idx, wt)
    for r in range(runs):
        src = [(s + 37 * r) % V for s in sources]
        got = en.run_batch(kinds, src)[0]
        for i, (k, s) in enumerate(zip(kinds, src)):
            assert np.array_equal(got[i], O.expected(og, k, s)), (r, i, k, s)


# A filter workgroup looks at 1024 vertices per step; from 33 workgroups on
# their completion is counted on several lines first.
@pytest.mark.parametrize("V", [1, 2, 1023, 1024, 1025, 32 * 1024, 32 * 1024 + 1, 40 * 1024 + 7])
@pytest.mark.parametrize("opts", [dict(frontier_dense_div=1), dict(frontier_dense_div=1 << 20),
                                  dict(sssp_delta=60)], ids=["sparse", "dense", "near_far"])
def test_filter_workgroups(gpu, V, opts):
    off, idx, wt = ring_graph(V, hub_degree=min(V // 2, 700))
    kinds = [BFS] * 3 + [SSSP] * 5 + [WCC]
    check(off, idx, wt, kinds, [0, V // 2, V - 1, V - 1, V // 3, 0, V // 2, V // 5, 0], runs=3, **opts)


# Batches of different mask widths in turn on one engine: the bits that mark
# vertices every BFS query has visited lie behind the pass's own records.
@pytest.mark.parametrize("V", [63, 64, 65, 127, 5001])
@pytest.mark.parametrize("div", [1, 1 << 20])
def test_mask_widths_in_turn(gpu, V, div):
    off, idx, wt = ring_graph(V, hub_degree=V // 3, chords=4)
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt), frontier_dense_div=div)
    og = O.G(off, idx, wt)
    for n in (150, 3, 70, 300, 1, 150):
        kinds = [BFS if i % 7 else SSSP for i in range(n)]
        src = [(i * 31 + n) % V for i in range(n)]
        got = en.run_batch(kinds, src)[0]
        for i, (k, s) in enumerate(zip(kinds, src)):
            assert np.array_equal(got[i], O.expected(og, k, s)), (n, i, k, s)


# Push work lists: vertices of at most 64 edges go 64 (or fewer) to a wave, of
# at most 2048 one to a wave or part of one, larger ones in chunks of 4096
# edges split into parts.  advance_blocks sets how many waves share the lists:
# one workgroup makes every list longer than the launch has waves.
@pytest.mark.parametrize("hub", [63, 64, 65, 2047, 2049, 4095, 4097, 9000])
@pytest.mark.parametrize("opts", [dict(), dict(advance_blocks=1), dict(advance_blocks=9, block_size=128),
                                  dict(advance_blocks=3, block_size=512, frontier_dense_div=1),
                                  dict(bin_small=1, bin_large=2), dict(sssp_delta=60)],
                         ids=["default", "one_block", "nine_blocks", "sparse", "all_large", "near_far"])
def test_push_work_lists(gpu, hub, opts):
    V = 12007
    off, idx, wt = ring_graph(V, hub_degree=hub, seed=hub, chords=2)
    check(off, idx, wt, [BFS, BFS, SSSP, SSSP], [V // 2, 0, V // 2, 5], runs=2, dense_threshold=65, **opts)


# The smallest launch the options allow, at every workgroup size (one 256-thread
# equivalent is half a workgroup of 512 threads).
@pytest.mark.parametrize("block", [128, 256, 512])
def test_smallest_advance_launch(gpu, block):
    off, idx, wt = ring_graph(5003, hub_degree=2500)
    check(off, idx, wt, [BFS, SSSP, SSSP], [0, 2501, 77], runs=2, advance_blocks=1, block_size=block)


# The same lists with two and four mask words, and on a directed graph.
@pytest.mark.parametrize("n", [5, 70, 150])
@pytest.mark.parametrize("directed", [False, True])
def test_push_mask_words(gpu, n, directed):
    V = 3001
    off, idx, wt = ring_graph(V, hub_degree=2500, seed=n, directed=directed)
    kinds = [SSSP] * (n // 3) + [BFS] * (n - n // 3)
    check(off, idx, wt, kinds, [(i * 131) % V for i in range(n)], runs=2, advance_blocks=2)


# Lane-per-query lists: claims of 1 to 64 items of at most 128 edges, items
# split down to 16 edges when the launch has more waves than items.  At most 16
# SSSP queries go to the narrow list (four edges per step), more to the wide
# one; dense_threshold=1 sends every SSSP word there.
@pytest.mark.parametrize("n", [1, 16, 17, 64, 70])
@pytest.mark.parametrize("hub", [15, 127, 129, 3000])
@pytest.mark.parametrize("opts", [dict(), dict(advance_blocks=1), dict(advance_blocks=9, frontier_dense_div=1),
                                  dict(dense_wide_addr=1, advance_blocks=2), dict(sssp_delta=60, advance_blocks=2),
                                  dict(dense_unroll=4)],
                         ids=["default", "one_block", "sparse", "wide_addr", "near_far", "unroll4"])
def test_lane_per_query_lists(gpu, n, hub, opts):
    V = 4099
    off, idx, wt = ring_graph(V, hub_degree=hub, seed=n, chords=2)
    check(off, idx, wt, [SSSP] * n + [BFS], [(i * 131) % V for i in range(n)] + [3], runs=2, dense_threshold=1,
          **opts)


# Weak components of directed graphs: below 4096 vertices every edge hooks, from
# there on after a sample of two out-edges per vertex.  Edges only enter the
# last vertices, and two parts stay apart.
@pytest.mark.parametrize("V", [4095, 4096, 4097, 70001])
def test_wcc_directed(gpu, V):
    rng = np.random.RandomState(V)
    half = V // 2
    top = half * 4 // 5  # no edge leaves the first part's vertices from here on
    a = np.concatenate([rng.randint(0, top, V), rng.randint(half, V, V // 3)])
    b = np.concatenate([rng.randint(0, half, V), rng.randint(half, V, V // 3)])
    keep = (a != b) & ((a < half) == (b < half))
    key = np.unique(a[keep].astype(np.int64) * V + b[keep])
    src, dst = key // V, key % V
    off = np.zeros(V + 1, np.int64)
    np.add.at(off, src + 1, 1)
    off = np.cumsum(off).astype(np.int32)
    got = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, dst.astype(np.int32))).wcc(2)
    exp = O.expected(O.G(off, dst.astype(np.int32), None), WCC, 0)
    assert np.array_equal(got[0], exp) and np.array_equal(got[1], exp)


# The same where the sample's rule turns: skewed graphs from as many edges as
# vertices on, others from four edges per vertex on and up to 2^18 vertices.
# Edges lead within sevenths of the vertices, so there are seven parts or more.
@pytest.mark.parametrize("V", [4096, 30011, 1 << 18, (1 << 18) + 1])
@pytest.mark.parametrize("per_vertex", [0.9, 1.1, 3.9, 4.1])
@pytest.mark.parametrize("hub", [False, True])
def test_wcc_directed_sample_rule(gpu, V, per_vertex, hub):
    rng = np.random.RandomState(V % 1000 + int(per_vertex * 10))
    n = int(V * per_vertex * 1.02) - (V // 7 if hub else 0)
    a = rng.randint(0, V, n).astype(np.int64)
    b = np.minimum(V - 1, a % 7 + 7 * rng.randint(0, V // 7, n))
    if hub:
        a = np.concatenate([a, np.full(V // 7, 7)])
        b = np.concatenate([b, np.arange(V // 7) * 7])
    keep = (a != b) & (a % 7 == b % 7)
    key = np.unique(a[keep] * V + b[keep])
    src, dst = key // V, key % V
    off = np.zeros(V + 1, np.int64)
    np.add.at(off, src + 1, 1)
    off, dst = np.cumsum(off).astype(np.int32), dst.astype(np.int32)
    got = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, dst)).wcc(1)[0]
    assert np.array_equal(got, O.expected(O.G(off, dst, None), WCC, 0))


# Near-far: pairs at or above the threshold wait in the far set.  Small and
# large steps, one to four mask words, BFS beside it, vertices without
# out-edges (a frontier that is empty while pairs wait), both frontier modes.
@pytest.mark.parametrize("delta", [1, 7, 60, 1000])
@pytest.mark.parametrize("n", [1, 5, 70, 200])
@pytest.mark.parametrize("opts", [dict(), dict(frontier_dense_div=1, dense_threshold=1),
                                  dict(frontier_dense_div=1 << 20, dense_threshold=1), dict(dense_threshold=65)],
                         ids=["default", "sparse_rows", "dense_rows", "edges"])
def test_near_far(gpu, delta, n, opts):
    V = 1501
    off, idx, wt = ring_graph(V, hub_degree=200, seed=n, chords=1)
    kinds = [SSSP] * n + [BFS] * (n // 2)
    check(off, idx, wt, kinds, [(i * 131) % V for i in range(len(kinds))], runs=2, sssp_delta=delta, **opts)


@pytest.mark.parametrize("delta", [1, 30])
def test_near_far_sinks(gpu, delta):
    # 0 -> 1..9 (sinks) at weight i, 0 -> 10 -> 11 -> ... at weight 90 each: when
    # only sinks are near the frontier has no edges and the path still waits.
    src = np.concatenate([np.zeros(10, np.int64), np.arange(10, 40)])
    dst = np.concatenate([np.arange(1, 11), np.arange(11, 41)])
    wt = np.concatenate([np.arange(1, 10), np.full(31, 90)]).astype(np.uint32)
    off = np.zeros(42, np.int64)
    np.add.at(off, src + 1, 1)
    check(np.cumsum(off).astype(np.int32), dst.astype(np.int32), wt, [SSSP, SSSP, BFS], [0, 10, 0], sssp_delta=delta)


@pytest.mark.parametrize("slots", [1, 4, 70])
def test_near_far_serving(gpu, slots):
    h = cgp_amd.HostCSR.grid(41, 37, p_extra=0.01, seed=3, wmin=1, wmax=1000)
    og = O.G.of(h)
    en = cgp_amd.Engine(cgp_amd.Graph.from_host(h), sssp_delta=300)
    en.serve_start(max_slots=slots)
    src = h.sample_sources(90, seed=2)
    for i, s in enumerate(src):
        en.serve_submit(SSSP if i % 3 else BFS, s, i, 0.0)
    left = set(range(len(src)))
    while left:
        for c in en.serve_step(max_iterations=3 if slots == 4 else 0):
            exp = O.expected(og, c["kind"], c["source"])
            assert np.array_equal(c["result"], exp), (c["ticket"], c["kind"], c["source"])
            left.remove(c["ticket"])
    en.serve_stop()


# Output of words that hold only BFS slots: straight from the depth planes while
# depths stay below 256 and V % 4 == 0 (a ring of V vertices has depths up to
# V / 2), through the value tile otherwise; 70 SSSP leave the second word mixed.
@pytest.mark.parametrize("V", [4, 28, 30, 400, 402, 511, 512, 600, 1028])
@pytest.mark.parametrize("n_sssp", [0, 3, 70])
@pytest.mark.parametrize("renumber", [False, True])
def test_bfs_output(gpu, V, n_sssp, renumber):
    off, idx, wt = ring_graph(V, chords=0 if V > 4 else 3)
    kinds = [BFS] * 150 + [SSSP] * n_sssp
    src = [(i * 7) % V for i in range(len(kinds))]
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt, renumber=renumber))
    og = O.G(off, idx, wt)
    exp = np.stack([O.expected(og, k, s) for k, s in zip(kinds, src)])
    assert np.array_equal(en.run_batch(kinds, src)[0], exp)
    # Device outputs at every alignment of a row start.
    buf = cgp_amd.DeviceBuffer((len(kinds) * V + 4) * 4)
    for shift in range(4):
        en.run_batch(kinds, src, out=buf.view(shift * 4, len(kinds) * V * 4))
        got = buf.to_host()[shift:shift + len(kinds) * V].reshape(len(kinds), V)
        assert np.array_equal(got, exp), shift


# The work counter of visited words: an edge of a frontier vertex reads one word
# per mask word with frontier bits there, unless every BFS query has visited its
# target and more than a sixteenth of the vertices are in that state (batch runs;
# allocation-free runs keep no such bits and read them all).
@pytest.mark.parametrize("n_bfs,n_sssp", [(1, 0), (40, 0), (100, 3), (200, 0)])
@pytest.mark.parametrize("div", [1, 1 << 20])
def test_visited_words_counted(gpu, n_bfs, n_sssp, div):
    V = 2003
    off, idx, wt = ring_graph(V, hub_degree=900, chords=4)
    src = [(i * 131) % V for i in range(n_bfs + n_sssp)]
    kinds = [BFS] * n_bfs + [SSSP] * n_sssp
    og = O.G(off, idx, wt)
    depth = np.stack([O.expected(og, BFS, s) for s in src[:n_bfs]]).astype(np.int64)
    word = (np.arange(n_bfs) + n_sssp) // 64  # SSSP queries take the first slots
    owner = np.repeat(np.arange(V), np.diff(off))
    last = depth.max(axis=0)
    every = read = 0
    for it in range(int(depth.max()) + 1):
        words = sum((depth[word == w] == it).any(axis=0).astype(np.int64) for w in range(word.max() + 1))
        done = last <= it
        edges = words[owner]
        every += int(edges.sum())
        read += int(edges[~done[idx]].sum()) if done.sum() > V // 16 else int(edges.sum())
    assert read < every
    en = cgp_amd.Engine(cgp_amd.Graph.from_csr(off, idx, wt), profile=2, frontier_dense_div=div)
    out = cgp_amd.DeviceBuffer(len(kinds) * V * 4)
    for _ in range(2):
        assert en.run_batch(kinds, src)[1]["work"][3] == read
    assert en.run_batch_static(kinds, src, out)["work"][3] == every


# The same two-level count in sparse mode: one vertex touches more than 32
# workgroups' share of vertices, fewer than the graph has, and each of those
# leads on.
@pytest.mark.parametrize("touched", [32 * 1024, 32 * 1024 + 1, 35000])
@pytest.mark.parametrize("n_bfs", [3, 70])
def test_filter_workgroups_of_a_touched_list(gpu, touched, n_bfs):
    V = 70001
    mid = 2 + (np.arange(touched) * 1.5).astype(np.int64)
    src = np.concatenate([[0], np.full(touched, 1), mid])
    dst = np.concatenate([[1], mid, mid + 1 + mid % 2 * 9000])
    off = np.zeros(V + 1, np.int64)
    np.add.at(off, src + 1, 1)
    wt = ((src * 7 + dst) % 13 + 1).astype(np.uint32)
    check(np.cumsum(off).astype(np.int32), dst.astype(np.int32), wt, [BFS] * n_bfs + [SSSP] * 2,
          [i % 2 for i in range(n_bfs + 2)], frontier_dense_div=1)
