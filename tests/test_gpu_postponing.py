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
