"""Multi-source BFS with two batches of 64 sources that walk the graph together:
source counts around one and two batches, every way a round is run, calls that
change between one mask and two on one preparation, levels that appear late.
Levels and digests against the CPU oracle, bit-exact."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu

PLANS = {"hbm": (1.0, 0), "zerocopy": (0.5, og.PLAN_ZERO_COPY), "zerocopy-eager": (0.5, og.PLAN_ZERO_COPY | og.PLAN_NO_GRAPH),
         "zerocopy-bins": (0.5, og.PLAN_ZERO_COPY | og.PLAN_NO_FUSE), "copy": (0.5, 0)}


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("plan", list(PLANS))
@pytest.mark.parametrize("V", [65, 4097, 30001])
def test_msbfs_pairs(V, plan, weighted):
    rng = np.random.default_rng(V)
    deg = rng.integers(0, 6, V)
    deg[0] = 5000
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    cols = rng.integers(0, V, E).astype(np.uint32)
    w = rng.integers(1, 64, E).astype(np.uint32) if weighted else None
    ptr = ptr[:-1].copy()
    g = og.Graph.from_csr(ptr, cols, w) if weighted else og.Graph.from_csr(ptr, cols)
    share, flags = PLANS[plan]
    full = (8 if weighted else 4) * E
    g.prepare("ascetic", edge_budget_bytes=max(64, int(full * share)), advisek=1.0 if share == 1 else 0.6, flags=flags,
              split_weight=16 if weighted else 0)
    pool = rng.integers(0, V, 24).astype(np.uint32)
    ref = {int(s): oracle.bfs(ptr, cols, int(s))[0] for s in set(pool.tolist())}
    sums = {s: og.levels_checksum(r) for s, r in ref.items()}
    for count, want in ((65, False), (3, True), (127, True), (128, False), (129, True), (64, False), (200, True)):
        src = rng.choice(pool, count)
        levels, got, reached, st = g.msbfs(src, want_levels=want)
        for i, s in enumerate(src.tolist()):
            assert int(got[i]) == sums[s], (count, i)
            assert int(reached[i]) == int((ref[s] != og.UNREACHED).sum())
            if want:
                assert np.array_equal(levels[i], ref[s]), (count, i)
        assert st["traversed_edges"] == sum(int(deg[ref[s] != og.UNREACHED].sum()) for s in src.tolist())
    g.close()
