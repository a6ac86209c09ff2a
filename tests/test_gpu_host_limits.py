"""What the library asks of the HIP runtime, seen and refused in between
(hip_shim): clears and the streams they go to, allocations that fail, memory
that stays."""
import pytest

import hip_shim

pytestmark = pytest.mark.gpu

PULL = """
def pull(V, seed=1):
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 9, V)
    deg[0] = 5
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    cols = rng.integers(0, V, int(ptr[-1])).astype(np.uint32)
    od = np.bincount(cols, minlength=V).astype(np.uint32)
    return ptr[:-1].copy(), cols, od
"""


def test_pagerank_clears_on_its_own_stream(gpu, tmp_path):
    """The arrival counters are cleared on the stream that counts in them (the
    others do not wait for the null stream), at the first run and after a tuning
    that takes more workgroups."""
    hip_shim.run(tmp_path, PULL + """
    ptr, cols, od = pull(40000)
    ref = oracle.pagerank(od, ptr, cols)[0]
    g = og.Graph.from_csr(ptr, cols, out_degree=od)
    for share in (1.0, 0.3):
        g.prepare("ascetic", edge_budget_bytes=int(4 * len(cols) * share), advisek=1.0 if share == 1 else 0.5)
        for t in (None, dict(t1=1, t2=2), dict(t1=1, t2=1)):
            if t:
                g.set_tuning(**t)
            null, mine = shim.shim_fills_null(), shim.shim_fills_stream()
            for fp64 in (False, True):
                assert np.abs(g.pagerank(fp64=fp64)[0] - ref).max() < 1e-6
            assert shim.shim_fills_null() == null
            if not t:
                assert shim.shim_fills_stream() > mine
    """)
