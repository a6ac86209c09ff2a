"""Rounds and loaders that the default plans of small graphs no longer reach.

In HBM, graphs above the one-launch rule (16384 vertices): every tuning, the
light/heavy split and bottom-up rounds, weighted and plain.  Out of memory, the
loader that gathers chunks into pinned slots and copies them (NO_FUSE without
ZERO_COPY): slots used again while earlier chunks are on their way, every
algorithm, packed and 8-byte edges, deferred orders and split rows.  All against
the oracle, bit-exact."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle
from test_gpu_tuning import TUNINGS

pytestmark = pytest.mark.gpu


def _source(ptr, E, k):
    return int(np.flatnonzero(np.diff(np.append(ptr.astype(np.int64), E)) > 0)[k])


@pytest.fixture(scope="module")
def rmat15():
    g = og.Graph.rmat(15, 16, seed=81, weight_seed=82)
    ptr, to, w, _ = g.export()
    src = _source(ptr, len(to), 7)
    yield g, ptr, to, w, src, oracle.bfs(ptr, to, src)[0], oracle.sssp(ptr, to, w, src), oracle.cc(ptr, to)[0]
    g.close()


@pytest.mark.parametrize("flags", [0, og.PLAN_NO_GRAPH, og.PLAN_NO_FUSE])
def test_tuning_in_hbm(gpu, rmat15, flags):
    g, ptr, to, w, src, bfs, sssp, cc = rmat15
    g.prepare("ascetic", edge_budget_bytes=8 * len(to), advisek=1.0, flags=flags)
    for t in TUNINGS:
        g.set_tuning(**t)
        for _ in range(2):
            assert np.array_equal(g.bfs(src)[0], bfs), t
            assert np.array_equal(g.sssp(src)[0], sssp), t
            assert np.array_equal(g.cc()[0], cc), t


@pytest.mark.parametrize("flags", [0, og.PLAN_NO_GRAPH])
@pytest.mark.parametrize("split,delta", [(32, 32), (8, 32), (8, 256), (40, 16), (16, 0)])
def test_split_in_hbm(gpu, rmat15, split, delta, flags):
    g, ptr, to, w, src, bfs, sssp, cc = rmat15
    g.prepare("ascetic", edge_budget_bytes=4 * len(to), advisek=1.0, flags=flags, split_weight=split)
    g.set_tuning(delta=delta)
    for _ in range(2):
        d, st = g.sssp(src)
        assert np.array_equal(d, sssp) and st["checksum"] == og.levels_checksum(d)
        assert np.array_equal(g.bfs(src)[0], bfs)
    assert np.array_equal(g.cc()[0], cc)


@pytest.mark.parametrize("flags", [0, og.PLAN_NO_GRAPH])
@pytest.mark.parametrize("graph", ["weighted", "er", "chain"])
def test_bottom_up_in_hbm(gpu, rmat15, graph, flags):
    """Bottom-up rounds on a weighted graph, on a dense one and after thousands of
    narrow rounds; node_sum is the level-synchronous oracle's."""
    own = graph != "weighted"
    if graph == "weighted":
        g = rmat15[0]
    elif graph == "er":
        g = og.Graph.er(20000, 24, seed=83)
    else:
        n = 18000
        src = np.concatenate([np.arange(2999), np.full(n - 3000, 2999)])
        g = og.Graph.from_edges(src, np.concatenate([np.arange(1, 3000), np.arange(3000, n)]), num_vertices=n + 5)
    ptr, to, w, _ = g.export()
    g.prepare("ascetic", edge_budget_bytes=(8 if w is not None else 4) * len(to), advisek=1.0,
              flags=flags | og.PLAN_DIRECTION_OPT)
    for s in (0 if graph == "chain" else _source(ptr, len(to), 7), _source(ptr, len(to), 1)):
        for _ in range(2):
            lv, st = g.bfs(s)
            ref, ns, _ = oracle.bfs(ptr, to, s)
            assert np.array_equal(lv, ref) and st["node_sum"] == ns
    if graph == "weighted":
        assert np.array_equal(g.sssp(rmat15[4])[0], rmat15[6])
    if own:
        g.close()


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("approach,frac,k", [("ascetic", 0.25, 0.8), ("ascetic", 1 / 64, 0.5), ("subway", 0.25, 0.0),
                                             ("subway", 1 / 64, 0.0)])
def test_gathered_chunks(gpu, rmat15, approach, frac, k, pack):
    g, ptr, to, w, src, bfs, sssp, cc = rmat15
    E, eb = len(to), 4 if pack else 8
    rng = np.random.default_rng(7)
    srcs = rng.choice(np.flatnonzero(np.diff(np.append(ptr.astype(np.int64), E)) > 0), 70).astype(np.uint32)
    for split in (0, 8) if pack else (0,):
        g.prepare(approach, edge_budget_bytes=int(E * eb * frac), advisek=k, split_weight=split,
                  flags=og.PLAN_NO_FUSE | (0 if pack else og.PLAN_NO_PACK))
        for _ in range(2):
            lv, st = g.bfs(src)
            assert np.array_equal(lv, bfs)
            assert st["gather_ms"] > 0 and st["h2d_bytes"] > 0 and st["h2d_bytes"] % eb == 0
            if frac < 0.1:  # more chunks than rounds and slots: each is used again in a round
                assert st["chunks"] > 4 * st["iterations"]
            labels, st = g.cc()
            assert np.array_equal(labels, cc) and st["gather_ms"] > 0
        for delta, defer in ((0, 0), (16, 0), (16, 1), (64, 2)):
            g.set_tuning(delta=delta, defer=defer)
            assert np.array_equal(g.sssp(src)[0], sssp), (split, delta, defer)
        g.set_tuning(defer=1)
        assert np.array_equal(g.cc()[0], cc)
        levels, sums, _, st = g.msbfs(srcs)
        assert st["gather_ms"] > 0
        for i in (0, 63, 64, 69):
            ref = oracle.bfs(ptr, to, int(srcs[i]))[0]
            assert np.array_equal(levels[i], ref) and sums[i] == og.levels_checksum(ref)


@pytest.mark.parametrize("frac", [0.25, 1 / 64])
def test_gathered_chunks_of_ids(gpu, rmat15, frac):
    """4-byte ids without weights."""
    _, ptr, to, _, src, bfs, _, cc = rmat15
    g = og.Graph.from_csr(ptr, to)
    g.prepare("ascetic", edge_budget_bytes=int(len(to) * 4 * frac), advisek=0.5, flags=og.PLAN_NO_FUSE)
    for _ in range(2):
        assert np.array_equal(g.bfs(src)[0], bfs)
        assert np.array_equal(g.cc()[0], cc)
        assert np.array_equal(g.msbfs([src, 0, 5])[0][0], bfs)
    g.close()
