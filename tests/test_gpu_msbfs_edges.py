"""Multi-source BFS at the edges of its groups: vertex counts around the 64 of a
wave, batches that are part-filled, full and one over, repeated sources, with
and without the levels (which take other kernels), twice in a row.  Levels and
digests against the CPU oracle, bit-exact."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("plan", ["hbm", "zerocopy", "copy"])
@pytest.mark.parametrize("count", [1, 64, 65])
@pytest.mark.parametrize("V", [1, 63, 64, 65, 4097, 70001])
def test_msbfs_groups(V, count, plan):
    rng = np.random.default_rng(V + count)
    deg = rng.integers(0, 6, V)
    deg[0] = min(V, 5000)
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    cols = rng.integers(0, V, int(ptr[-1])).astype(np.uint32)
    ptr = ptr[:-1].copy()
    src = rng.integers(0, V, count).astype(np.uint32)
    g = og.Graph.from_csr(ptr, cols)
    budget, k = (4 * len(cols), 1.0) if plan == "hbm" else (max(64, len(cols)), 0.5)
    g.prepare("ascetic", edge_budget_bytes=budget, advisek=k, flags=og.PLAN_ZERO_COPY if plan == "zerocopy" else 0)
    ref = {int(s): oracle.bfs(ptr, cols, int(s))[0] for s in set(src.tolist())}
    for want in (False, True, False):
        levels, sums, reached, st = g.msbfs(src, want_levels=want)
        for i, s in enumerate(src):
            r = ref[int(s)]
            assert int(sums[i]) == og.levels_checksum(r)
            assert int(reached[i]) == int((r != og.UNREACHED).sum())
            if want:
                assert np.array_equal(levels[i], r)
        edges = np.asarray(deg, np.int64)
        assert st["traversed_edges"] == sum(int(edges[ref[int(s)] != og.UNREACHED].sum()) for s in src)
    g.close()
