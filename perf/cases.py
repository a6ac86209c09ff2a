"""The work that users of this framework have it do, as cases that can be timed.

A case is one call (or one burst of queries) through the Python binding on a
graph that the program has loaded and prepared before: the traversals, connected
components, PageRank, the multi-source batch, the allocation-free entry point
and the query server.  Graphs are the two families of bench.py and the tests,
drawn from the seed on the GPU: directed R-MAT (.57/.19/.19/.05, loops and
repeated arcs removed, weights uniform in [1, 63]) cut to any vertex count, and
undirected Erdos-Renyi.  Sources are vertices with out-edges.

The programs here have torch in their process, whose HIP runtime (7.0) refuses
the event nodes that the engine records into captured rounds; such programs
prepare their graphs with PLAN_NO_GRAPH, and so do these cases.
"""
import math

import numpy as np
import torch

import onegraph_amd as og

RMAT = (0.57, 0.19, 0.19)


def listed():
    return [
        # A traversal of a small graph, as in a test suite or an interactive
        # tool: launches and latency are all there is.
        dict(name="bfs small", path="bfs", vertices=5000, degree=16, plan="hbm"),
        # The allocation-free entry point over arrays that are on the device
        # already, in a mid-sized graph.
        dict(name="bfs device arrays", path="bfs_device", vertices=150001, degree=16),
        # The in-memory configuration of the benchmark: R-MAT scale 20.
        dict(name="bfs in memory", path="bfs", vertices=1 << 20, degree=16, plan="hbm"),
        # Direction-optimising BFS, a larger graph of odd size.
        dict(name="bfs direction-optimising", path="bfs", vertices=1500007, degree=16, plan="diropt"),
        # Out of memory with gathered chunks copied to the device.
        dict(name="bfs copied chunks", path="bfs", vertices=1000003, degree=16, plan="copy", budget=0.25,
             advisek=0.8, approach="ascetic"),
        # Shortest paths on a graph in memory, settings of the query lanes.
        dict(name="sssp in memory", path="sssp", vertices=400009, degree=16, plan="hbm", split=8, delta=256),
        # The headline configuration: a quarter of the edge bytes on the
        # device, the rest read over the link.
        dict(name="sssp out of memory", path="sssp", vertices=1 << 24, degree=16, plan="zerocopy", budget=0.25,
             advisek=0.8, split=8, delta=256),
        # Connected components out of memory, the benchmark's plan on a
        # smaller graph of the same family with some vertices apart.
        dict(name="cc out of memory", path="cc", vertices=3000001, degree=32, plan="zerocopy", budget=0.25,
             advisek=0.8),
        # PageRank in FP64 on a graph with hubs that fits.
        dict(name="pagerank fp64 in memory", path="pagerank", vertices=300007, degree=16, family="rmat", fp64=True,
             budget=1.0, advisek=1.0),
        # PageRank in FP32 out of memory, the benchmark's plan.
        dict(name="pagerank out of memory", path="pagerank", vertices=3000001, degree=32, family="er", fp64=False,
             budget=0.25, advisek=0.8),
        # Many sources at once, out of memory, digests only: the batch of the
        # benchmark (two full masks of 64) on a smaller graph.
        dict(name="bfs many sources", path="msbfs", vertices=1 << 22, degree=16, sources=128, levels=False,
             plan="zerocopy", budget=0.5, advisek=0.8),
        # A burst of queries at the server, seven in ten BFS.
        dict(name="served queries", path="serve", vertices=1 << 19, degree=16, bfs=70, sssp=30),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["bfs", "bfs", "bfs_device", "bfs_copy", "sssp", "sssp_ooc", "cc", "pagerank", "msbfs", "serve"])
    degree = rng.randint(6, 24)
    if path == "bfs":
        return dict(path="bfs", vertices=_log(rng, 1 << 11, 1 << 21), degree=degree, plan=rng.choice(["hbm", "diropt"]))
    if path == "bfs_device":
        return dict(path=path, vertices=_log(rng, 1 << 11, 1 << 21), degree=degree)
    if path == "bfs_copy":
        return dict(path="bfs", vertices=_log(rng, 1 << 15, 1 << 21), degree=degree, plan="copy",
                    budget=round(rng.uniform(0.1, 0.5), 3), advisek=round(rng.uniform(0.3, 0.9), 3),
                    approach=rng.choice(["ascetic", "subway"]))
    if path == "sssp":
        split = rng.choice([0, 8])
        return dict(path="sssp", vertices=_log(rng, 1 << 11, 1 << 21), degree=degree, plan="hbm", split=split,
                    delta=256 if split else 32)
    if path == "sssp_ooc":
        split = rng.choice([0, 8])
        return dict(path="sssp", vertices=_log(rng, 1 << 16, 1 << 22), degree=degree, plan="zerocopy",
                    budget=round(rng.uniform(0.15, 0.5), 3), advisek=0.8, split=split, delta=256 if split else 32)
    if path == "cc":
        budget = rng.choice([0.25, 0.5, 1.0])
        return dict(path="cc", vertices=_log(rng, 1 << 12, 3 << 20), degree=rng.randint(3, 32),
                    plan="hbm" if budget == 1.0 else "zerocopy", budget=budget, advisek=1.0 if budget == 1.0 else 0.8)
    if path == "pagerank":
        budget = rng.choice([0.25, 1.0])
        return dict(path="pagerank", vertices=_log(rng, 1 << 12, 3 << 20), degree=degree,
                    family=rng.choice(["rmat", "er"]), fp64=rng.random() < 0.5, budget=budget,
                    advisek=1.0 if budget == 1.0 else 0.8)
    if path == "msbfs":
        levels = rng.random() < 0.3  # whole level arrays: V values for every source, so smaller graphs
        return dict(path="msbfs", vertices=_log(rng, 1 << 12, 1 << (17 if levels else 22)), degree=degree,
                    sources=rng.randint(1, 128), levels=levels, plan="zerocopy", budget=rng.choice([0.5, 1.0]),
                    advisek=0.8)
    bfs = rng.randint(4, 70)
    return dict(path="serve", vertices=_log(rng, 1 << 13, 1 << 19), degree=degree, bfs=bfs, sssp=rng.randint(1, 30))


# ------------------------------------------------------------------ graphs


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _arcs(family, n, degree, gen, dev, apart=False):
    """Distinct arcs without loops, sorted by (source, target), as one int64
    key source * n + target."""
    if family == "er":  # n * degree / 2 undirected edges, both directions
        m = n * degree // 2
        u = torch.randint(0, n, (m,), generator=gen, device=dev)
        v = torch.randint(0, n, (m,), generator=gen, device=dev)
        keep = u != v
        if apart:  # one vertex in 16 has no arcs
            lone = torch.rand(n, generator=gen, device=dev) < 1 / 16
            keep &= ~(lone[u] | lone[v])
        u, v = u[keep], v[keep]
        key = torch.cat([u * n + v, v * n + u])
    else:
        a, b, c = RMAT
        u = torch.zeros(n * degree, dtype=torch.int64, device=dev)
        v = torch.zeros_like(u)
        for _ in range(max(1, (n - 1).bit_length())):
            r = torch.rand(u.shape, generator=gen, device=dev)
            down = r >= a + b
            right = ((r >= a) & ~down) | (r >= a + b + c)
            u = 2 * u + down
            v = 2 * v + right
        keep = (u != v) & (u < n) & (v < n)
        key = u[keep] * n + v[keep]
    return torch.unique(key)  # sorted


def _rows(src, n):
    """Row offsets (n + 1) of arcs sorted by source."""
    deg = torch.bincount(src, minlength=n)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=src.device)
    torch.cumsum(deg, 0, out=ptr[1:])
    return ptr, deg


def _u32(t):
    return t.to(torch.int32).cpu().numpy().view(np.uint32)


def _csr(case, seed):
    """Out-edge CSR on the device: offsets, targets, weights, degrees."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    n = case["vertices"]
    family = case.get("family", "er" if case["path"] == "cc" else "rmat")
    key = _arcs(family, n, case["degree"], gen, dev, apart=case["path"] == "cc")
    src = key // n
    dst = key - src * n
    ptr, deg = _rows(src, n)
    w = torch.randint(1, 64, dst.shape, generator=gen, device=dev) if case["path"] in ("sssp", "serve") else None
    return ptr, src, dst, w, deg


def _host_graph(case, seed):
    ptr, _, dst, w, deg = _csr(case, seed)
    g = og.Graph.from_csr(ptr[:-1].cpu().numpy().view(np.uint64), _u32(dst), None if w is None else _u32(w))
    return g, deg.cpu().numpy()


def _prepared(g, case):
    """Places the graph as bench.py does for the plan that the case names."""
    E = g.num_edges
    plan = case.get("plan", "hbm")
    split = case.get("split", 0)
    eb = 8 if case["path"] in ("sssp", "serve") else 4
    flags = og.PLAN_NO_GRAPH | {"diropt": og.PLAN_DIRECTION_OPT, "zerocopy": og.PLAN_ZERO_COPY}.get(plan, 0)
    if plan in ("hbm", "diropt"):
        g.prepare("ascetic", edge_budget_bytes=E * eb, advisek=1.0, flags=flags, split_weight=split)
    else:
        g.prepare(case.get("approach", "ascetic"), edge_budget_bytes=max(1, int(E * eb * case["budget"])),
                  advisek=case["advisek"], flags=flags, split_weight=split)
    if "delta" in case:
        g.set_tuning(delta=case["delta"])


def _sources(deg, count, seed):
    cand = np.flatnonzero(deg > 0)
    return np.random.default_rng(seed).choice(cand, count, replace=count > len(cand)).astype(np.uint32)


# ------------------------------------------------------------------- cases


def prepare(case, seed):
    path = case["path"]
    if path == "bfs_device":
        ptr, _, dst, _, deg = _csr(case, seed)
        n = case["vertices"]
        return dict(case=case, ptr=ptr, cols=dst.to(torch.int32), source=int(_sources(deg.cpu().numpy(), 1, seed)[0]),
                    levels=torch.empty(n, dtype=torch.int32, device=ptr.device))
    if path == "pagerank":
        ptr, src, dst, _, deg = _csr(case, seed)
        n = case["vertices"]
        order = torch.argsort(dst, stable=True)
        iptr, _ = _rows(dst[order], n)
        g = og.Graph.from_csr(iptr[:-1].cpu().numpy().view(np.uint64), _u32(src[order]), out_degree=_u32(deg))
        g.prepare("ascetic", edge_budget_bytes=int(g.num_edges * 4 * case["budget"]), advisek=case["advisek"])
        return dict(case=case, graph=g)
    g, deg = _host_graph(case, seed)
    if path == "serve":
        g.prepare("ascetic", edge_budget_bytes=g.num_edges * 8, advisek=1.0,
                  flags=og.PLAN_NO_GRAPH | og.PLAN_DIRECTION_OPT, split_weight=8)
        g.set_tuning(delta=256)
        src = _sources(deg, case["bfs"] + case["sssp"], seed)
        kinds = np.random.default_rng(seed + 1).permutation(
            [og.QUERY_BFS] * case["bfs"] + [og.QUERY_SSSP] * case["sssp"])
        return dict(case=case, graph=g, server=og.Server([g]),
                    queries=[(int(k), int(s)) for k, s in zip(kinds, src)])
    _prepared(g, case)
    if path == "cc":
        return dict(case=case, graph=g)
    return dict(case=case, graph=g, sources=_sources(deg, case.get("sources", 1), seed))


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "bfs_device":
        n = case["vertices"]
        st = og.bfs_device_noalloc(state["ptr"].data_ptr(), state["cols"].data_ptr(), n, state["cols"].numel(),
                                   state["source"], state["levels"].data_ptr())
        return dict(levels=state["levels"], reached=st["reached"], edges=st["traversed_edges"])
    g = state["graph"]
    if path in ("bfs", "sssp"):
        values, st = (g.bfs if path == "bfs" else g.sssp)(int(state["sources"][0]))
        return dict(values=values, reached=st["reached"], edges=st["traversed_edges"])
    if path == "cc":
        return g.cc()[0]
    if path == "pagerank":
        return g.pagerank(fp64=case["fp64"])[0]
    if path == "msbfs":
        levels, sums, reached, st = g.msbfs(state["sources"], want_levels=case["levels"])
        out = dict(checksums=sums.view(np.int64), reached=reached.view(np.int64), edges=st["traversed_edges"])
        if case["levels"]:
            out["levels"] = levels
        return out
    srv = state["server"]
    # the program wants the whole arrays of one query in 16, else the digests
    ids = [srv.submit(0, kind, source, keep=i % 16 == 0) for i, (kind, source) in enumerate(state["queries"])]
    got = {}
    while len(got) < len(ids):
        for r in srv.poll(4096, timeout_ms=1000):
            got[r["id"]] = r
    rows = [got[i] for i in ids]
    return dict(values=[srv.take_values(i, 0) for i in ids[::16]],
                checksums=np.array([r["checksum"] for r in rows], np.uint64).view(np.int64),
                counts=np.array([[r["status"], r["reached"], r["traversed_edges"]] for r in rows], np.int64))


def work(case):
    """Each row offset, edge and result once; for queries once per traversal
    (a batch of 64 sources shares its edge reads)."""
    n = case["vertices"]
    m = n * case["degree"]
    path = case["path"]
    eb = 8 if path in ("sssp", "serve") else 4
    if path == "pagerank":
        return dict(bytes=8 * n + 4 * m + 4 * n + (8 if case["fp64"] else 4) * n, flops=m)
    one = 8 * n + eb * m + 4 * n
    if path == "msbfs":
        batches = (case["sources"] + 63) // 64
        return dict(bytes=batches * (8 * n + 4 * m) + case["sources"] * (4 * n if case["levels"] else 16), flops=0)
    if path == "serve":
        return dict(bytes=((case["bfs"] + 63) // 64) * (8 * n + 4 * m) + case["sssp"] * one, flops=0)
    return dict(bytes=one, flops=0)


def exact(case, seed):
    """PageRank by its definition in FP64; the others are whole numbers."""
    if case["path"] != "pagerank":
        return None
    _, src, dst, _, deg = _csr(case, seed)
    n = case["vertices"]
    deg = deg.double()
    dangling = deg == 0
    rank = torch.full((n,), 1.0 / n, dtype=torch.float64, device=src.device)
    for _ in range(100):
        share = torch.where(dangling, 0.0, rank / deg.clamp(min=1))
        got = torch.zeros_like(rank).index_add_(0, dst, share[src])
        new = 0.15 / n + 0.85 * (got + rank[dangling].sum() / n)
        change = (new - rank).abs().sum().item()
        rank = new
        if change < 1e-7:
            break
    return rank
