"""The compaction's wide form, which reserves the dynamic list's places under a
lock: many workgroups at once, one and four windows each, in rounds that read
in place, gather chunks and hold vertices back.  Against the oracle, and the
same rounds as the one-word form."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [og.PLAN_ZERO_COPY, og.PLAN_ZERO_COPY | og.PLAN_NO_GRAPH, og.PLAN_NO_FUSE])
@pytest.mark.parametrize("V", [5, 4097, 300001, (1 << 22) + 3])
def test_wide_lists(gpu, V, flags):
    rng = np.random.default_rng(V)
    deg = rng.integers(0, 5, V).astype(np.int64)
    deg[0] = min(V, 300)
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    cols, w = rng.integers(0, V, E).astype(np.uint32), rng.integers(1, 64, E).astype(np.uint32)
    ptr = ptr[:-1].copy()
    g = og.Graph.from_csr(ptr, cols, w)
    bfs, sssp = oracle.bfs(ptr, cols, 0)[0], oracle.sssp(ptr, cols, w, 0)
    counts = []
    for wide in (og.PLAN_TEST_WIDE_LISTS, 0):
        plan = g.prepare("ascetic", edge_budget_bytes=max(16, E), advisek=0.5, flags=flags | wide, split_weight=8)
        assert plan["vsplit"] < V
        for _ in range(2):
            lv, st = g.bfs(0)
            assert np.array_equal(lv, bfs)
            counts.append([st[k] for k in ("iterations", "node_sum", "static_node_sum", "work_edges", "checksum")])
        for delta, defer in ((0, 0), (64, 0), (64, 2)):
            g.set_tuning(delta=delta, defer=defer)
            assert np.array_equal(g.sssp(0)[0], sssp), (wide, delta, defer)
        assert np.array_equal(g.cc()[0], oracle.cc(ptr, cols)[0])
        assert np.array_equal(g.msbfs([0, V - 1])[0][0], bfs)
    assert all(c == counts[0] for c in counts)
    g.close()
