"""PageRank's chunk ring counts what it used: every iteration moves the dynamic
region once, whether the run ends at its limit, where nothing is copied
beyond it, or by its residual, where the ring had gone on into the next one."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,frac", [(257, 0.3), (5001, 0.02), (5001, 0.3), (200003, 0.05), (200003, 0.5)])
def test_ring_counts(gpu, V, frac):
    rng = np.random.default_rng(V)
    deg = rng.integers(0, 40, V)
    deg[0] = 5
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    cols = rng.integers(0, V, E).astype(np.uint32)
    od = np.bincount(cols, minlength=V).astype(np.uint32)
    g = og.Graph.from_csr(ptr[:-1].copy(), cols, out_degree=od)
    plan = g.prepare("ascetic", edge_budget_bytes=max(4 * 160, int(4 * E * frac)), advisek=0.5)
    assert plan["vsplit"] < V
    edges = E - int(ptr[plan["vsplit"]])
    one = g.pagerank(max_iterations=1)[1]["run"]
    # narrow words of the bits of V - 1, chunks rounded up to words
    bits = (V - 1).bit_length()
    assert bits * edges <= 8 * one["h2d_bytes"] <= bits * edges + 128 * one["chunks"]
    for limit in (2, 3, 100):
        r, st = g.pagerank(max_iterations=limit)
        n = st["iterations"]
        assert n == limit or (limit == 100 and n < 100)
        assert st["run"]["chunks"] == n * one["chunks"], (limit, n)
        assert st["run"]["h2d_bytes"] == n * one["h2d_bytes"], (limit, n)
    assert np.abs(r - oracle.pagerank(od, ptr[:-1], cols)[0]).max() < 1e-6
    g.close()
