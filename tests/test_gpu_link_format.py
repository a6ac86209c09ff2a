"""Dynamic regions that cross the link as narrow words: every path that reads
them (zero-copy rounds with and without the light/heavy split, multi-source
BFS, PageRank's chunk ring), at id widths of 1 to 17 bits, weights of 1 to 6
bits and up to 2^20 (too wide for narrow words), rows that end anywhere in a
word, and slots down to a few edges.  Integers bit-exact against the oracle,
PageRank within the repository's 1e-6 of FP64."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu


def _graph(V, seed, wmax):
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 9, V)
    deg[0] = 5
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    return ptr[:-1].copy(), rng.integers(0, V, E).astype(np.uint32), rng.integers(1, wmax + 1, E).astype(np.uint32)


@pytest.mark.parametrize("approach", ["ascetic", "subway"])
@pytest.mark.parametrize("wmax", [1, 63, 1 << 20])
@pytest.mark.parametrize("V", [2, 3, 17, 256, 257, 5001, 70001])
def test_zero_copy_narrow_words(V, wmax, approach):
    ptr, cols, w = _graph(V, V + wmax, wmax)
    E = len(cols)
    plain = og.Graph.from_csr(ptr, cols)
    plain.prepare(approach, edge_budget_bytes=max(16, E), advisek=0.5, flags=og.PLAN_ZERO_COPY)
    assert np.array_equal(plain.bfs(0)[0], oracle.bfs(ptr, cols, 0)[0])
    assert np.array_equal(plain.cc()[0], oracle.cc(ptr, cols)[0])
    src = np.arange(min(V, 3), dtype=np.uint32)
    levels = plain.msbfs(src)[0]
    for i, s in enumerate(src):
        assert np.array_equal(levels[i], oracle.bfs(ptr, cols, int(s))[0])
    plain.close()
    g = og.Graph.from_csr(ptr, cols, w)
    ref = oracle.sssp(ptr, cols, w, 0)
    for split in (0, 8) if wmax < 64 else (0,):  # (the split needs packed edges)
        g.prepare(approach, edge_budget_bytes=max(16, E), advisek=0.5, flags=og.PLAN_ZERO_COPY, split_weight=split)
        g.set_tuning(delta=16)
        assert np.array_equal(g.sssp(0)[0], ref)
        assert np.array_equal(g.bfs(0)[0], oracle.bfs(ptr, cols, 0)[0])
    g.close()


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("frac", [0.02, 0.3, 1.0])
@pytest.mark.parametrize("V", [3, 257, 5001, 70001])
def test_pagerank_chunk_ring(V, frac, fp64):
    ptr, cols, _ = _graph(V, V, 1)
    E = len(cols)
    od = np.bincount(cols, minlength=V).astype(np.uint32)  # cols are the in-neighbours
    g = og.Graph.from_csr(ptr, cols, out_degree=od)
    # (never below two slots of the longest row, 8 edges)
    g.prepare("ascetic", edge_budget_bytes=max(4 * 40, int(4 * E * frac)), advisek=1.0 if frac == 1.0 else 0.5)
    ref, it, _ = oracle.pagerank(od, ptr, cols)
    for _ in range(2):
        r, st = g.pagerank(fp64=fp64)
        assert np.abs(r.astype(np.float64) - ref).max() < 1e-6
        assert abs(st["iterations"] - it) <= 1
    assert g.pagerank(fp64=fp64, max_iterations=3)[1]["iterations"] == 3
    g.close()


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("approach", ["ascetic", "subway"])
def test_copy_loader(approach, pack):
    """The copy loader, which reads pinned rows in place, and with NO_OVERLAP
    gathers and copies them: rounds that relax a few rows and most of the dynamic
    region, 5000 empty rows in a stretch, a row that spans several workgroups
    (9000 edges).  Both against the oracle, and the same rounds and edges."""
    V = 30001
    rng = np.random.default_rng(5)
    deg = rng.integers(0, 9, V)
    deg[15000:20000] = 0
    deg[21000] = 9000
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    cols = rng.integers(0, V, int(ptr[-1])).astype(np.uint32)
    w = rng.integers(1, 64, len(cols)).astype(np.uint32)
    ptr = ptr[:-1].copy()
    base = 0 if pack else og.PLAN_NO_PACK
    src = 21000
    bfs, sssp, cc = oracle.bfs(ptr, cols, src)[0], oracle.sssp(ptr, cols, w, src), oracle.cc(ptr, cols)[0]
    for weights, eb in ((None, 4), (w, 8)):
        g = og.Graph.from_csr(ptr, cols, weights)
        for split in (0, 8) if weights is not None and pack else (0,):
            counts = []
            for flags in (base, base | og.PLAN_NO_OVERLAP, base | og.PLAN_NO_GRAPH):
                g.prepare(approach, edge_budget_bytes=len(cols) * eb // 2, advisek=0.5, flags=flags, split_weight=split)
                for _ in range(2):
                    g.set_tuning(delta=0)
                    assert np.array_equal(g.cc()[0], cc)
                    lv, st = g.bfs(src)
                    assert np.array_equal(lv, bfs)
                    counts.append([st[k] for k in ("iterations", "node_sum", "work_edges", "reached", "checksum")])
                    assert st["chunks"] > 0 and st["h2d_bytes"] > 0
                    assert np.array_equal(g.msbfs(np.array([src, 0], np.uint32))[0][0], bfs)
                    if weights is not None:
                        for delta in (0, 16):
                            g.set_tuning(delta=delta)
                            assert np.array_equal(g.sssp(src)[0], sssp)
            assert all(c == counts[0] for c in counts)
        g.close()
