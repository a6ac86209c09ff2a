"""Small graphs, which one workgroup traverses in one launch: vertex counts at
the edges of its bitmaps (32), of its sweep (1024, 4096) and of the rule that
takes a graph there (8192 for CC, 16384), edge counts at the rule's limit
(196608), rows at the edges of its bins (0, 32, 512).  Results against the CPU
oracle and the general rounds, bit-exact."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu

LIMIT = 3 << 16


def _graph(V, E, seed):
    """Rows of 0..2, 31..33, 511..513 edges and one hub that takes what is left
    of E; the graph's far end is reached over a path."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 3, V).astype(np.int64)
    for k, d in enumerate((0, 31, 32, 33, 511, 512, 513)):
        deg[(V // 2 + k) % V] = d
    deg[V - 1] = 1
    while deg.sum() > E:
        deg[rng.integers(0, V)] = 0
    deg[V // 3] += E - deg.sum()
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    return ptr[:-1].copy(), rng.integers(0, V, E).astype(np.uint32), rng.integers(1, 64, E).astype(np.uint32), V // 3


@pytest.mark.parametrize("E", [0, 20000, LIMIT, LIMIT + 1])
@pytest.mark.parametrize("V", [1, 31, 32, 33, 1023, 1025, 4096, 4097, 8192, 8193, 16383, 16384, 16385])
def test_small_edges(V, E):
    E = E or 4 * V
    ptr, cols, w, src = _graph(V, E, V + E)
    g = og.Graph.from_csr(ptr, cols, w)
    want = {"bfs": oracle.bfs(ptr, cols, src)[0], "sssp": oracle.sssp(ptr, cols, w, src), "cc": oracle.cc(ptr, cols)[0]}
    for flags, split in ((0, 0), (og.PLAN_NO_GRAPH, 0), (og.PLAN_NO_FUSE, 0), (og.PLAN_NO_PACK, 0), (0, 16)):
        g.prepare("ascetic", edge_budget_bytes=8 * E, advisek=1.0, flags=flags, split_weight=split)
        stats = []
        for _ in range(2):
            lv, st = g.bfs(src)
            assert np.array_equal(lv, want["bfs"]), (flags, split)
            stats.append([st[k] for k in ("iterations", "node_sum", "static_node_sum", "work_edges", "reached",
                                          "traversed_edges", "checksum")])
            assert np.array_equal(g.sssp(src)[0], want["sssp"]), (flags, split)
            assert np.array_equal(g.cc()[0], want["cc"]), (flags, split)
        assert stats[0] == stats[1]
        if flags == og.PLAN_NO_GRAPH:
            small = stats[0]
        if flags == og.PLAN_NO_FUSE:  # the general rounds count the same
            assert stats[0] == small
    g.close()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("V,E", [(1, 1), (33, 200), (4097, 30000), (16384, LIMIT), (16385, LIMIT), (16384, LIMIT + 1)])
def test_small_device_arrays(gpu, V, E, shift):
    """The entry over device arrays, with levels at any word of an allocation;
    wrong offsets are refused with the levels untouched."""
    ptr, cols, _, src = _graph(V, E, V + 3 * E)
    hip = _Hip()
    try:
        full = np.append(ptr, np.uint64(E)).astype(np.uint64)
        off = full.copy()
        off[0] = 1
        d_ptr, d_off, d_cols = hip.upload(full), hip.upload(off), hip.upload(cols)
        lv = hip.upload(np.full(V + 2 + shift, 77, np.uint32))
        at = lv + 4 * shift
        with pytest.raises(og.OgError):
            og.bfs_device_noalloc(d_off, d_cols, V, E, src, at)
        assert (hip.download(lv, np.uint32, V + 2 + shift) == 77).all()
        want = oracle.bfs(ptr, cols, src)[0]
        for _ in range(2):
            st = og.bfs_device_noalloc(d_ptr, d_cols, V, E, src, at)
            got = hip.download(lv, np.uint32, V + 2 + shift)
            assert np.array_equal(got[shift:shift + V], want)
            assert (got[shift + V:] == 77).all() and (got[:shift] == 77).all()
            assert st["reached"] == int((want != og.UNREACHED).sum())
    finally:
        hip.free()
