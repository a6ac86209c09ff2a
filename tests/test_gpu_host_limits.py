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


def test_runs_after_a_refused_allocation(gpu, tmp_path):
    """A first call that runs out of memory part of the way fails with that
    status, and the next one, with memory, is whole: PageRank's state and the two
    chunks of results above 8 MB."""
    hip_shim.run(tmp_path, PULL + """
    V = (1 << 21) + 5
    ptr, cols, od = pull(V)
    ref = oracle.pagerank(od, ptr, cols)[0]
    g = og.Graph.from_csr(ptr, cols, out_degree=od)
    g.prepare("ascetic", edge_budget_bytes=4 * len(cols), advisek=1.0)

    def refused(deny, lo, hi, name, call):
        before = shim.shim_denied()
        deny(lo, hi)
        try:
            call()
            raise SystemExit("not refused")
        except og.OgError as e:
            assert e.name == name, e
        finally:
            deny(1, 0)
        assert shim.shim_denied() > before

    refused(shim.shim_deny_device, 8 * V, 8 * V, "OG_ENOMEM_DEVICE", g.pagerank)   # ranks, contributions
    refused(shim.shim_deny_device, 4 * V, 4 * V, "OG_ENOMEM_DEVICE", g.pagerank)   # out-degrees
    refused(shim.shim_deny_pinned, 8 << 20, 8 << 20, "OG_ENOMEM_HOST", lambda: g.pagerank(fp64=True))
    for fp64 in (True, False):
        assert np.abs(g.pagerank(fp64=fp64)[0] - ref).max() < 1e-6
    """)
