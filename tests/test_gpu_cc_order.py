"""CC's orders over the two regions (og_tuning.defer): a path of 2000 vertices in
the static region, whose smallest label takes a round a hop or so to its far
end, and leaves in the dynamic region that hang on that end.  Both regions
every round (2) relaxes the leaves in the first round and again as labels
arrive; held back until the path has settled (0, 1) they relax once."""
import numpy as np
import pytest

import onegraph_amd as og
import oracle

pytestmark = pytest.mark.gpu

PATH, LEAVES = 2000, 3000


@pytest.fixture(scope="module")
def graph():
    p, leaf = np.arange(PATH - 1), PATH + np.arange(LEAVES)
    end = np.full(LEAVES, PATH - 1)
    g = og.Graph.from_edges(np.concatenate([p, end]), np.concatenate([p + 1, leaf]), symmetrize=True)
    yield g
    g.close()


@pytest.mark.parametrize("flags", [og.PLAN_ZERO_COPY, og.PLAN_ZERO_COPY | og.PLAN_NO_GRAPH, og.PLAN_NO_FUSE])
def test_orders(gpu, graph, flags):
    ptr, cols, _, _ = graph.export()
    plan = graph.prepare("ascetic", edge_budget_bytes=4 * 7800, advisek=0.95, flags=flags)
    held = graph.num_vertices - plan["vsplit"]
    assert plan["vsplit"] >= PATH and held > LEAVES // 2
    want = oracle.cc(ptr, cols)[0]
    assert graph.tuning()["defer"] == 0
    seen = {}
    for defer in (None, 0, 1, 2):
        if defer is not None:
            graph.set_tuning(defer=defer)
        labels, st = graph.cc()
        assert np.array_equal(labels, want), defer
        seen[defer] = st["node_sum"] - st["static_node_sum"]
    assert seen[None] == seen[0] == seen[1] == held
    assert seen[2] >= 2 * held


def test_autotuner_knows_the_orders(gpu, graph):
    ptr, cols, _, _ = graph.export()
    graph.prepare("ascetic", edge_budget_bytes=4 * 7800, advisek=0.95, flags=og.PLAN_ZERO_COPY)
    best, ms = graph.autotune(og.TUNE_CC, runs=1)
    assert best["defer"] in (0, 1, 2) and ms > 0 and graph.tuning() == best
    assert np.array_equal(graph.cc()[0], oracle.cc(ptr, cols)[0])
