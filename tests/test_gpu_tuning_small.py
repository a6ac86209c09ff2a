"""The autotuner on graphs that are traversed in one launch, which no tuning
shapes: the installed tuning stays.  The rounds are tuned as before."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu

MINE = dict(t1=5, lpv0=32, t2=77, tile=128, delta=9, defer=0, dyn_grid=3)


def _graph(V, E, seed):
    rng = np.random.default_rng(seed)
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(np.bincount(rng.integers(0, V, E), minlength=V))
    return ptr[:-1].copy(), rng.integers(0, V, E).astype(np.uint32), rng.integers(1, 64, E).astype(np.uint32)


@pytest.mark.parametrize("algo,V", [(og.TUNE_BFS, 16384), (og.TUNE_SSSP, 16384), (og.TUNE_CC, 8192)])
def test_autotune_keeps_the_tuning_of_one_launch(gpu, algo, V):
    ptr, cols, w = _graph(V, 60000, algo + 1)
    src = int(np.argmax(np.diff(np.append(ptr, np.uint64(len(cols))).astype(np.int64))))
    g = og.Graph.from_csr(ptr, cols, w)
    g.prepare("ascetic", edge_budget_bytes=8 * len(cols), advisek=1.0)
    g.set_tuning(**MINE)
    best, ms = g.autotune(algo, src, runs=1)
    assert best == MINE and g.tuning() == MINE and ms > 0
    assert np.array_equal(g.sssp(src)[0], oracle.sssp(ptr, cols, w, src))
    # the multi-source search has rounds on such a graph too
    g.autotune(og.TUNE_MSBFS, 1, runs=1)
    assert np.array_equal(g.msbfs([src])[0][0], oracle.bfs(ptr, cols, src)[0])
    g.close()


def test_autotune_tunes_the_rounds_of_a_small_graph(gpu):
    """OG_PLAN_NO_FUSE keeps the rounds, and with them the tuning."""
    ptr, cols, w = _graph(16384, 60000, 5)
    g = og.Graph.from_csr(ptr, cols, w)
    g.prepare("ascetic", edge_budget_bytes=8 * len(cols), advisek=1.0, flags=og.PLAN_NO_FUSE)
    g.set_tuning(**MINE)
    best, _ = g.autotune(og.TUNE_BFS, int(cols[0]), runs=1)
    assert g.tuning() == best
    assert np.array_equal(g.bfs(0)[0], oracle.bfs(ptr, cols, 0)[0])
    g.close()
