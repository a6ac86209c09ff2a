"""Frontier compaction at the edges of its windows: vertex counts around 4, 4096
and 2^22 (where a workgroup takes four windows instead of one), rows of every
bin in one graph, held-back and deferred vertices.  Results against the CPU
oracle, bit-exact."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 4, 5, 63, 4095, 4096, 4097, 16385, (1 << 22) + 3]


def _graph(V, seed):
    """Rows of 0-2 edges, some of 40-100 (bin 1) and one hub (bin 2 from
    V = 5000 on), targets uniform: every window holds flagged vertices."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 3, V).astype(np.int64)
    deg[rng.integers(0, V, max(1, V // 1000))] = rng.integers(40, 100)
    deg[V // 3] = min(V, 9000)
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    return ptr[:-1].copy(), rng.integers(0, V, E).astype(np.uint32), rng.integers(1, 64, E).astype(np.uint32), V // 3


@pytest.mark.parametrize("plan", ["hbm", "zerocopy"])
@pytest.mark.parametrize("V", SIZES)
def test_compaction_window_edges(V, plan):
    ptr, cols, w, src = _graph(V, 100 + V % 97)
    E = len(cols)
    if E == 0:
        pytest.skip("no edges")
    g = og.Graph.from_csr(ptr, cols, w)
    budget, k, flags = (E * 8, 1.0, 0) if plan == "hbm" else (max(64, E * 2), 0.6, og.PLAN_ZERO_COPY)
    big = V > 100000
    for split in ((8,) if big else (0, 8)):
        g.prepare("ascetic", edge_budget_bytes=budget, advisek=k, flags=flags, split_weight=split)
        assert np.array_equal(g.bfs(src)[0], oracle.bfs(ptr, cols, src)[0])
        ref = oracle.sssp(ptr, cols, w, src)
        for delta, defer in ((0, 0), (16, 0), (16, 1), (16, 2)) if not big else ((64, 1),):
            g.set_tuning(delta=delta, defer=defer)
            assert np.array_equal(g.sssp(src)[0], ref), (split, delta, defer)
        for defer in (0, 1):
            g.set_tuning(defer=defer)
            assert np.array_equal(g.cc()[0], oracle.cc(ptr, cols)[0]), (split, defer)
    g.close()


@pytest.mark.parametrize("flags", [0, og.PLAN_NO_GRAPH, og.PLAN_NO_FUSE, og.PLAN_NO_OVERLAP, og.PLAN_ZERO_COPY])
@pytest.mark.parametrize("weights", ["light", "heavy", "at the split", "mixed"])
def test_heavy_rounds_follow_at_once(weights, flags):
    """Light/heavy split: a light round that puts nothing below the threshold is
    followed by the heavy round.  Paths (every round has one vertex) beside a
    random graph, edges of one kind only and of both, buckets below, at and above
    the split, deferred orders (which keep the empty sweep)."""
    V, split = 20011, 8
    rng = np.random.default_rng(3)
    deg = rng.integers(0, 5, V)
    deg[:300] = 1  # a path of 300
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    cols = rng.integers(0, V, E).astype(np.uint32)
    cols[:300] = np.arange(1, 301)
    lo, hi = {"light": (1, split), "heavy": (split, 64), "at the split": (split - 1, split + 1), "mixed": (1, 64)}[weights]
    w = rng.integers(lo, hi, E).astype(np.uint32)
    w[-1] = 63
    ptr = ptr[:-1].copy()
    ref = oracle.sssp(ptr, cols, w, 0)
    g = og.Graph.from_csr(ptr, cols, w)
    for share in (1.0, 0.3):
        g.prepare("ascetic", edge_budget_bytes=int(8 * E * share), advisek=1.0 if share == 1 else 0.5,
                  flags=flags if share < 1 else flags & ~og.PLAN_ZERO_COPY, split_weight=split)
        for delta in (1, 8, 256):
            for defer in (0, 1, 2):
                g.set_tuning(delta=delta, defer=defer)
                assert np.array_equal(g.sssp(0)[0], ref), (share, delta, defer)
    g.close()
