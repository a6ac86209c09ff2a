"""Results on their way to the host: sizes at the edges of the slabs (32 KiB), of
the single-threaded copy (256 KiB) and of the staging (8 MiB), FP64 ranks (twice
the bytes), results that fill part of a caller's array, and several graphs
whose results leave at once (one takes the staging, the others go round it)."""
import threading

import numpy as np
import pytest

import onegraph_amd as og

pytestmark = pytest.mark.gpu


def _ring(V):
    """0 -> 1, 2, 3 and v -> v - 1: level 2 for 1..3, the rest unreached."""
    ptr = np.arange(V, dtype=np.uint64) + 2
    ptr[0] = 0
    cols = np.concatenate([np.arange(1, 4, dtype=np.uint32), np.arange(V - 1, dtype=np.uint32)])
    ptr[1:] = 3 + np.arange(V - 1)
    return og.Graph.from_csr(ptr, cols)


def _expect(V):
    want = np.full(V, og.UNREACHED, np.uint32)
    want[0] = 1
    want[1:4] = 2
    return want


@pytest.mark.parametrize("flags", [0, og.PLAN_NO_GRAPH])
@pytest.mark.parametrize("V", [5, 8191, 8192, 8193, 65536, 65537, 1 << 20, (1 << 21) - 1, 1 << 21, (1 << 21) + 1])
def test_result_sizes(V, flags):
    g = _ring(V)
    g.prepare("ascetic", edge_budget_bytes=4 * g.num_edges, advisek=1.0, flags=flags)
    want = _expect(V)
    for _ in range(2):
        assert np.array_equal(g.bfs(0)[0], want)
    g.close()


@pytest.mark.parametrize("V", [8193, 40000, (1 << 20) + 3])
def test_fp64_ranks(V):
    ptr = np.arange(V, dtype=np.uint64)
    g = og.Graph.from_csr(ptr, (np.arange(V, dtype=np.uint32) + 1) % V, out_degree=np.ones(V, np.uint32))
    g.prepare("ascetic", edge_budget_bytes=4 * V, advisek=1.0)
    assert np.allclose(g.pagerank(fp64=True)[0], 1 / V, rtol=1e-12)  # a cycle: uniform ranks
    g.close()


@pytest.mark.parametrize("share", [1.0, 0.5])
@pytest.mark.parametrize("fp64", [False, True])
def test_ranks_not_wanted(fp64, share):
    """Statistics alone: nothing after the iterations waits for the stream."""
    V = 40000
    ptr = 8 * np.arange(V, dtype=np.uint64)
    cols = ((np.arange(8 * V) * 7) % V).astype(np.uint32)
    g = og.Graph.from_csr(ptr, cols, out_degree=np.bincount(cols, minlength=V).astype(np.uint32))
    g.prepare("ascetic", edge_budget_bytes=int(32 * V * share), advisek=1.0 if share == 1 else 0.5)
    for _ in range(5):
        r, st = g.pagerank(fp64=fp64, want_values=False)
        assert r is None and st["iterations"] == g.pagerank(fp64=fp64)[1]["iterations"]
    g.close()


def test_results_leave_at_once():
    sizes = [1 << 20, 65537, 300001, (1 << 21) + 1]
    graphs = [_ring(V) for V in sizes]
    for g in graphs:
        g.prepare("ascetic", edge_budget_bytes=4 * g.num_edges, advisek=1.0, flags=og.PLAN_NO_GRAPH)
    bad = []

    def work(g, V):
        want = _expect(V)
        for _ in range(20):
            if not np.array_equal(g.bfs(0)[0], want):
                bad.append(V)

    threads = [threading.Thread(target=work, args=a) for a in zip(graphs, sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for g in graphs:
        g.close()
