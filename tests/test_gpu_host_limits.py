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
    hip_shim.run(tmp_path, PULL, """
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
    hip_shim.run(tmp_path, PULL, """
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


LINK = """
def graph(V, weighted, seed=3):
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 9, V)
    deg[0] = 5
    ptr = np.zeros(V + 1, np.uint64)
    ptr[1:] = np.cumsum(deg)
    E = int(ptr[-1])
    cols, w = rng.integers(0, V, E).astype(np.uint32), rng.integers(1, 64, E).astype(np.uint32)
    return og.Graph.from_csr(ptr[:-1].copy(), cols, w if weighted else None), ptr, cols, w

def link_bytes(ptr, plan, bits):   # of the narrow words of the dynamic region
    n = int(ptr[-1] - ptr[plan["vsplit"]])
    return ((n * bits + 31) // 32 + 2) * 4, 4 * n
"""


def test_link_format_only_where_it_is_read(gpu, tmp_path):
    """The narrow copy of the dynamic region is built for rounds that read it, in
    place of the packed words; loaders that gather chunks hold whole edges only."""
    hip_shim.run(tmp_path, LINK, """
    V = 70001
    for weighted, bits in ((False, 17), (True, 23)):
        g, ptr, cols, w = graph(V, weighted)
        E = len(cols)
        for flags, split in ((0, 0), (og.PLAN_ZERO_COPY, 0), (og.PLAN_ZERO_COPY | og.PLAN_NO_OVERLAP, 0),
                             (og.PLAN_NO_OVERLAP, 0), (og.PLAN_NO_FUSE, 0)) + (((0, 8),) if weighted else ()):
            plan = g.prepare("ascetic", edge_budget_bytes=2 * E, advisek=0.5, flags=flags, split_weight=split)
            narrow, whole = link_bytes(ptr, plan, bits)
            in_place = flags & og.PLAN_ZERO_COPY or not flags
            assert shim.shim_pinned_has(narrow) == bool(in_place), (weighted, flags)
            if weighted:
                assert shim.shim_pinned_has(whole) == (not in_place), flags
            assert np.array_equal(g.bfs(0)[0], oracle.bfs(ptr[:-1], cols, 0)[0]), (weighted, flags)
            if weighted:
                assert np.array_equal(g.sssp(0)[0], oracle.sssp(ptr[:-1], cols, w, 0)), flags
        g.close()
    """)


def test_no_memory_for_the_link_format(gpu, tmp_path):
    """Without pinned memory for the narrow words the edges cross as they are."""
    hip_shim.run(tmp_path, LINK, PULL, """
    V = 70001
    for weighted, bits in ((False, 17), (True, 23)):
        g, ptr, cols, w = graph(V, weighted)
        for flags, split in ((0, 0), (og.PLAN_ZERO_COPY, 0)) + (((0, 8),) if weighted else ()):
            plan = g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5, flags=flags, split_weight=split)
            narrow, whole = link_bytes(ptr, plan, bits)
            before = shim.shim_denied()
            shim.shim_deny_pinned(narrow, narrow)
            g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5, flags=flags, split_weight=split)
            shim.shim_deny_pinned(1, 0)
            assert shim.shim_denied() == before + 1
            for _ in range(2):
                lv, st = g.bfs(0)
                assert np.array_equal(lv, oracle.bfs(ptr[:-1], cols, 0)[0])
                assert st["h2d_bytes"] % 4 == 0 and st["h2d_bytes"] > 0
                assert np.array_equal(g.cc()[0], oracle.cc(ptr[:-1], cols)[0])
                if weighted:
                    g.set_tuning(delta=16)
                    assert np.array_equal(g.sssp(0)[0], oracle.sssp(ptr[:-1], cols, w, 0))
        g.close()
    ptr, cols, od = pull(V)
    g = og.Graph.from_csr(ptr, cols, out_degree=od)
    plan = g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
    narrow, whole = link_bytes(np.append(ptr, np.uint64(len(cols))), plan, 17)
    before = shim.shim_denied()
    shim.shim_deny_pinned(narrow, narrow)
    g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
    shim.shim_deny_pinned(1, 0)
    assert shim.shim_denied() == before + 1
    assert np.abs(g.pagerank()[0] - oracle.pagerank(od, ptr, cols)[0]).max() < 1e-6
    """)


def test_no_memory_for_the_result_staging(gpu, tmp_path):
    """Results up to 8 MB leave through pinned staging of 256 KiB or 8 MiB and
    flags of 2 KiB; without any one of them they leave through the runtime, from
    the one-launch traversal too.  Preparing and running do not fail, and
    staging is used again once there is memory."""
    hip_shim.run(tmp_path, LINK, """
    for size in (256 << 10, 8 << 20, 2048):
        for V in (3000, 70001, 300001):
            g, ptr, cols, w = graph(V, True)
            ref = oracle.bfs(ptr[:-1], cols, 0)[0], oracle.sssp(ptr[:-1], cols, w, 0)
            before = shim.shim_denied()
            shim.shim_deny_pinned(size, size)
            g.prepare("ascetic", edge_budget_bytes=8 * len(cols), advisek=1.0)
            for _ in range(2):
                assert np.array_equal(g.bfs(0)[0], ref[0])
                assert np.array_equal(g.sssp(0)[0], ref[1])
            if size == 2048 or (size == 256 << 10) == (4 * V <= 256 << 10):
                assert shim.shim_denied() > before, (size, V)
            shim.shim_deny_pinned(1, 0)
            assert np.array_equal(g.bfs(0)[0], ref[0])
            g.close()       # (the process's staging goes with the last preparation)
    """)


def test_missing_slabs_are_an_error(gpu, tmp_path):
    """A result whose slabs do not come (the export is left out, the stream
    reports an error once and synchronises without) is an error, not an array
    with holes."""
    hip_shim.run(tmp_path, LINK, """
    V = 300001
    g, ptr, cols, w = graph(V, False)
    g.prepare("ascetic", edge_budget_bytes=4 * len(cols), advisek=1.0)
    ref = oracle.bfs(ptr[:-1], cols, 0)[0]
    assert np.array_equal(g.bfs(0)[0], ref)
    shim.shim_skip_launch((4 * V + 32767) // 32768, 256)
    shim.shim_query_error(1)
    try:
        g.bfs(0)
        raise SystemExit("no error")
    except og.OgError as e:
        assert e.name == "OG_EHIP", e
    shim.shim_skip_launch(0, 0)
    shim.shim_query_error(0)
    for _ in range(3):
        assert np.array_equal(g.bfs(0)[0], ref)
    """)


def test_host_threads_bound_result_copies(gpu, tmp_path):
    """Results of 1.2 MB: with host_threads = 1 no threads are kept for them, with
    4 three helpers beside the caller."""
    hip_shim.run(tmp_path, LINK, """
    import os
    V = 300001
    g, ptr, cols, w = graph(V, False)
    ref = oracle.bfs(ptr[:-1], cols, 0)[0]

    def threads_with(n):
        g.prepare("ascetic", edge_budget_bytes=4 * len(cols), advisek=1.0, host_threads=n)
        for _ in range(3):
            assert np.array_equal(g.bfs(0)[0], ref)
        return len(os.listdir("/proc/self/task"))

    threads_with(1)     # (the runtime's own threads are there now)
    one = threads_with(1)
    assert threads_with(4) == one + 3
    assert threads_with(2) == one + 3   # (one pool for the process)
    assert threads_with(1) == one
    """)


def test_multi_source_state_of_one_width(gpu, tmp_path):
    """A preparation that has served short and long batches holds the state of the
    widest, not of both: 48 bytes a vertex, with levels 128 more, beside what is
    independent of the graph (2048 workgroups' sums, the turned levels).  Replayed
    rounds follow the state when it moves."""
    hip_shim.run(tmp_path, LINK, """
    V = 300001
    g, ptr, cols, w = graph(V, False)
    rng = np.random.default_rng(5)
    src = rng.choice(np.flatnonzero(np.diff(ptr.astype(np.int64)) > 0), 100).astype(np.uint32)
    ref = np.array([oracle.bfs(ptr[:-1], cols, int(s))[0] for s in src])
    sums = np.array([og.levels_checksum(r) for r in ref], np.uint64)
    fixed = 2 * 2048 * 3 * 64 * 8 + (1 << 16)
    for budget, k, flags in ((4 * len(cols), 1.0, 0), (2 * len(cols), 0.5, og.PLAN_ZERO_COPY)):
        for order in ((30, 100, 64, 65, 30), (100, 1, 100)):
            g.prepare("ascetic", edge_budget_bytes=budget, advisek=k, flags=flags)
            assert np.array_equal(g.msbfs(src[:0], want_levels=False)[1], sums[:0])
            base = shim.shim_live_device()
            for n in order:
                for _ in range(2):
                    assert np.array_equal(g.msbfs(src[:n], want_levels=False)[1], sums[:n]), n
            assert shim.shim_live_device() - base <= 48 * V + fixed, (shim.shim_live_device() - base) / V
            for n in order:
                for _ in range(2):
                    lv, cs, _, _ = g.msbfs(src[:n])
                    assert np.array_equal(lv, ref[:n]) and np.array_equal(cs, sums[:n]), n
                    assert np.array_equal(g.msbfs(src[:n], want_levels=False)[1], sums[:n]), n
            assert shim.shim_live_device() - base <= (48 + 128 + 4 * 64) * V + fixed
    """)


def test_graph_in_pageable_memory(gpu, tmp_path):
    """A graph that could not be pinned: traversals gather chunks and need the
    slots alone pinned, PageRank copies from where the edges are; zero-copy is
    refused."""
    hip_shim.run(tmp_path, LINK, PULL, """
    V = 70001
    E = graph(V, False)[1][-1]
    shim.shim_deny_pinned(int(4 * E), int(4 * E))
    g, ptr, cols, w = graph(V, False)
    shim.shim_deny_pinned(1, 0)
    try:
        g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5, flags=og.PLAN_ZERO_COPY)
        raise SystemExit("not refused")
    except og.OgError as e:
        assert e.name == "OG_EUNSUPPORTED", e
    plan = g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
    narrow, whole = link_bytes(ptr, plan, 17)
    before = shim.shim_denied()
    shim.shim_deny_pinned(narrow, narrow)
    g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
    assert shim.shim_denied() == before
    shim.shim_deny_pinned(1, 0)
    for _ in range(2):
        lv, st = g.bfs(0)
        assert np.array_equal(lv, oracle.bfs(ptr[:-1], cols, 0)[0]) and st["gather_ms"] > 0
        assert np.array_equal(g.cc()[0], oracle.cc(ptr[:-1], cols)[0])
    ptr, cols, od = pull(V)
    shim.shim_deny_pinned(4 * len(cols), 4 * len(cols))
    g = og.Graph.from_csr(ptr, cols, out_degree=od)
    shim.shim_deny_pinned(1, 0)
    ref = oracle.pagerank(od, ptr, cols)[0]
    for deny in (0, 1):
        plan = g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
        if deny:
            narrow, whole = link_bytes(np.append(ptr, np.uint64(len(cols))), plan, 17)
            shim.shim_deny_pinned(narrow, narrow)
            g.prepare("ascetic", edge_budget_bytes=2 * len(cols), advisek=0.5)
            shim.shim_deny_pinned(1, 0)
        for _ in range(2):
            assert np.abs(g.pagerank()[0] - ref).max() < 1e-6
    """)


def test_levels_with_little_memory(gpu, tmp_path):
    """Level arrays leave the device for up to 64 sources at a time, for fewer
    where there is no memory for that."""
    hip_shim.run(tmp_path, LINK, """
    V = 70001
    g, ptr, cols, w = graph(V, False)
    src = np.arange(70, dtype=np.uint32)
    ref = np.array([oracle.bfs(ptr[:-1], cols, int(s))[0] for s in src])
    for n, room in ((64, 64), (70, 128)):   # the levels take 64 or 128 bytes a vertex, 64 turned ones 256
        g.prepare("ascetic", edge_budget_bytes=4 * len(cols), advisek=1.0)
        g.msbfs(src[:n], want_levels=False)
        before = shim.shim_denied()
        shim.shim_deny_device(room * V + 1, 1 << 40)
        for _ in range(2):
            assert np.array_equal(g.msbfs(src[:n])[0], ref[:n])
        shim.shim_deny_device(1, 0)
        assert shim.shim_denied() > before
    """)
