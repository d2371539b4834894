"""The engine's workloads as timed cases: one call of a public entry point each.

A case names an algorithm (`algo`: bfs, sssp, pagerank, mbfs), a graph family (`graph`) with its
sizes, and the options of the call.  prepare() draws the graph from the seed on the GPU, uploads
it as a program does (medusa_amd.Graph from host CSR arrays) and keeps the handle and an output
buffer; run() is one call.  Every algorithm runs with its default options unless the case says
otherwise.
"""
import math

import numpy as np
import torch

import medusa_amd as md

DEV = "cuda"
DAMPING = 0.85


def listed():
    return [
        # the smallest calls a program makes: a traversal of a few thousand vertices into host memory,
        # where launches and waits are all there is
        dict(name="bfs_er4k", algo="bfs", graph="er", n=4096, m=32768, host_out=True),
        # BFS on a mid-size uniform graph (the reference's first configuration: 65,536 / 1,048,576)
        dict(name="bfs_er64k", algo="bfs", graph="er", n=65536, m=1048576),
        # the benchmark's power-law graph, BFS from its largest hub: few, wide supersteps
        dict(name="bfs_rmat20", algo="bfs", graph="rmat", scale=20, edge_factor=16),
        # a sparse power-law graph with a long tail of thin supersteps (2.4 M vertices, 5 M arcs)
        dict(name="bfs_chung_lu", algo="bfs", graph="chung_lu", n=2400000, m=5000000),
        # many independent graphs packed into one handle, one source each
        dict(name="bfs_batch", algo="bfs", graph="batch", count=64, lo_log2=10, hi_log2=16, edge_factor=8),
        # route lengths on a small and on a large road-like network, odd sides and even
        dict(name="sssp_lattice_small", algo="sssp", graph="lattice", rows=173, cols=211),
        dict(name="sssp_lattice", algo="sssp", graph="lattice", rows=1400, cols=1400),
        # weighted distances on the power-law graph (uint32 weights 1..1000)
        dict(name="sssp_rmat20", algo="sssp", graph="rmat", scale=20, edge_factor=16),
        # ranking a mid-size graph, launched superstep by superstep
        dict(name="pagerank_rmat16", algo="pagerank", graph="rmat", scale=16, edge_factor=16, steps=30,
             use_graph=False),
        # the headline: 30 supersteps of a million vertices, captured as one graph
        dict(name="pagerank_rmat20", algo="pagerank", graph="rmat", scale=20, edge_factor=16, steps=30,
             use_graph=True),
        # every graph of a batch ranked in the same launches
        dict(name="pagerank_batch", algo="pagerank", graph="batch", count=64, lo_log2=10, hi_log2=16, edge_factor=8,
             steps=20, use_graph=True),
        # 64 traversals at once as bit masks (all-pairs samples, centrality)
        dict(name="mbfs_rmat20", algo="mbfs", graph="rmat", scale=20, edge_factor=16, k=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    algo = rng.choice(["bfs", "bfs", "sssp", "pagerank", "pagerank", "mbfs"])
    if algo == "sssp":
        family = rng.choice(["er", "rmat", "lattice", "lattice"])
    elif algo == "mbfs":
        family = rng.choice(["er", "rmat", "chung_lu"])
    else:
        family = rng.choice(["er", "rmat", "chung_lu", "batch"])
    c = dict(algo=algo, graph=family)
    if family == "er":
        n = _log_int(rng, 4096, 1 << 20)
        c.update(n=n, m=n * rng.randint(8, 16) + rng.randint(0, 999))
    elif family == "rmat":
        c.update(scale=rng.randint(12, 20), edge_factor=rng.randint(8, 16))
    elif family == "chung_lu":
        n = _log_int(rng, 4096, 1000000 if algo == "mbfs" else 2400000)
        c.update(n=n, m=int(n * rng.uniform(2.0, 4.0)))
    elif family == "batch":
        c.update(count=rng.randint(8, 64), lo_log2=10, hi_log2=rng.randint(13, 16), edge_factor=rng.randint(4, 8))
    else:
        c.update(rows=_log_int(rng, 60, 1400), cols=_log_int(rng, 60, 1400))
    if algo == "pagerank":
        c.update(steps=rng.randint(10, 30), use_graph=rng.random() < 0.5)
    elif algo == "mbfs":
        c.update(k=rng.randint(1, 64))
    elif algo == "bfs":
        c.update(host_out=rng.random() < 0.25)
    return c


# ---- graphs: arcs (src, dst, weight-or-None) on the GPU, from the seed alone -----------------


def _er(g, n, m):
    src = torch.randint(0, n, (m,), generator=g, device=DEV)
    dst = torch.randint(0, n, (m,), generator=g, device=DEV)
    keep = src != dst
    return src[keep], dst[keep]


def _rmat(g, scale, m, a=0.45, b=0.15, c=0.15, noise=0.1):
    """Quadrant probabilities a/b/c/d, each scaled by 1 +- noise per arc and level and renormalised."""
    src = torch.zeros(m, dtype=torch.int64, device=DEV)
    dst = torch.zeros(m, dtype=torch.int64, device=DEV)
    quad = torch.tensor([a, b, c, 1.0 - a - b - c], device=DEV).view(4, 1)
    for _ in range(scale):
        p = quad * (1.0 + noise * (2.0 * torch.rand((4, m), generator=g, device=DEV) - 1.0))
        edge = p.cumsum(0)
        r = torch.rand(m, generator=g, device=DEV) * edge[3]
        row = r >= edge[1]
        col = torch.where(row, r >= edge[2], r >= edge[0])
        src = (src << 1) | row
        dst = (dst << 1) | col
    return src, dst


def _chung_lu(g, n, m, exponent=2.0, p_zero=0.4):
    """Zipf out-weights (40 % of the vertices have none), destinations uniform."""
    top = min(100000, n - 1)
    cdf = torch.arange(1, top + 1, device=DEV, dtype=torch.float64).pow(-exponent).cumsum(0)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    w = (torch.searchsorted(cdf, u) + 1).clamp_(max=top)
    w[torch.rand(n, generator=g, device=DEV) < p_zero] = 0
    cum = w.cumsum(0)
    x = (torch.rand(m, generator=g, device=DEV, dtype=torch.float64) * cum[-1]).long()
    src = torch.searchsorted(cum, x, right=True).clamp_(max=n - 1)
    return src, torch.randint(0, n, (m,), generator=g, device=DEV)


def _lattice(g, rows, cols, p_keep=0.7, p_diag=0.02):
    """Right and down edges kept with p_keep, one diagonal per cell with p_diag, both directions,
    one weight per undirected edge."""
    ids = torch.arange(rows * cols, device=DEV).view(rows, cols)
    pick = lambda shape, p: torch.rand(shape, generator=g, device=DEV) < p  # noqa: E731
    h, v = pick((rows, cols - 1), p_keep), pick((rows - 1, cols), p_keep)
    d, left = pick((rows - 1, cols - 1), p_diag), pick((rows - 1, cols - 1), 0.5)
    right, anti = d & ~left, d & left
    a = torch.cat([ids[:, :-1][h], ids[:-1][v], ids[:-1, :-1][right], ids[:-1, 1:][anti]])
    b = torch.cat([ids[:, 1:][h], ids[1:][v], ids[1:, 1:][right], ids[1:, :-1][anti]])
    w = torch.randint(1, 1001, (len(a),), generator=g, device=DEV)
    return torch.cat([a, b]), torch.cat([b, a]), torch.cat([w, w])


def _arcs(case, seed):
    """(n, src, dst, weight-or-None, graph starts): arcs sorted by source, stable."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    family, w = case["graph"], None
    if family == "er":
        n, (src, dst) = case["n"], _er(g, case["n"], case["m"])
    elif family == "rmat":
        n = 1 << case["scale"]
        src, dst = _rmat(g, case["scale"], case["edge_factor"] * n)
    elif family == "chung_lu":
        n, (src, dst) = case["n"], _chung_lu(g, case["n"], case["m"])
    elif family == "lattice":
        n = case["rows"] * case["cols"]
        src, dst, w = _lattice(g, case["rows"], case["cols"])
    else:  # batch: independent Chung-Lu graphs, sizes evenly spread over their logarithm
        sizes = [int(x) for x in np.exp2(np.linspace(case["lo_log2"], case["hi_log2"], case["count"]))]
        begin = np.concatenate([[0], np.cumsum(sizes)])
        parts = [_chung_lu(g, k, case["edge_factor"] * k) for k in sizes]
        src = torch.cat([s + int(b) for (s, _), b in zip(parts, begin)])
        dst = torch.cat([d + int(b) for (_, d), b in zip(parts, begin)])
        n = int(begin[-1])
    if case["algo"] == "sssp" and w is None:
        w = torch.randint(1, 1001, (len(src),), generator=g, device=DEV)
    src, order = torch.sort(src, stable=True)
    starts = begin if family == "batch" else np.array([0, n])
    return n, src, dst[order], None if w is None else w[order], starts


def _out_degree(n, src):
    return torch.bincount(src, minlength=n)


def _sources(case, seed, outdeg, starts):
    """The reference's root rule (the vertex of largest out-degree, of every graph of a batch), the
    middle of a lattice, k random vertices with out-edges for the masks."""
    if case["algo"] == "mbfs":
        cand = torch.nonzero(outdeg).flatten().cpu().numpy()
        rs = np.random.default_rng(seed)
        return np.sort(rs.choice(cand, size=min(case["k"], len(cand)), replace=False)).astype(np.uint32)
    if case["graph"] == "lattice":
        return np.array([case["rows"] // 2 * case["cols"] + case["cols"] // 2], np.uint32)
    deg = outdeg.cpu().numpy()
    return np.array([b + int(np.argmax(deg[b:e])) for b, e in zip(starts[:-1], starts[1:])], np.uint32)


# ---- one call ---------------------------------------------------------------------------------


def prepare(case, seed):
    n, src, dst, w, starts = _arcs(case, seed)
    outdeg = _out_degree(n, src)
    row_ptr = np.zeros(n + 1, np.uint32)
    row_ptr[1:] = outdeg.cumsum(0).cpu().numpy()
    host = lambda t: None if t is None else t.to(torch.int32).cpu().numpy().view(np.uint32)  # noqa: E731
    graph = md.Graph(row_ptr, host(dst), host(w))
    if len(starts) > 2:
        graph.set_batch(starts)
    state = dict(case=case, graph=graph)
    algo = case["algo"]
    if algo != "pagerank":
        state["sources"] = _sources(case, seed, outdeg, starts)
    if algo == "mbfs":
        state["out"] = torch.empty((len(state["sources"]), n), dtype=torch.uint8, device=DEV)
    elif case.get("host_out"):
        state["out"] = np.empty(n, np.int32)
    else:
        dtype = {"bfs": torch.int32, "sssp": torch.uint32, "pagerank": torch.float32}[algo]
        state["out"] = torch.empty(n, dtype=dtype, device=DEV)
    torch.cuda.synchronize()
    return state


def run(state):
    case, graph, out = state["case"], state["graph"], state["out"]
    algo = case["algo"]
    if algo == "pagerank":
        rank, st = graph.pagerank(DAMPING, case["steps"], out=out, use_graph=int(case["use_graph"]))
        return {"rank": rank, "residual": st.residual_l1}
    if algo == "mbfs":
        levels, st = graph.mbfs(state["sources"], out=out)
        return {"levels": levels, "reached": st.reached, "edges": st.edges_traversed}
    if algo == "sssp":
        dist, st = graph.sssp(int(state["sources"][0]), out=out)
        return {"dist": dist.view(torch.int32), "reached": st.reached, "edges": st.edges_traversed}
    if case["graph"] == "batch":
        levels, st = graph.bfs_multi(state["sources"], out=out)
    else:
        levels, st = graph.bfs(int(state["sources"][0]), out=out)
    return {"levels": levels, "reached": st.reached, "edges": st.edges_traversed}


def _size(case):
    """Vertices and arcs (expected, for the random families)."""
    family = case["graph"]
    if family == "rmat":
        return 1 << case["scale"], case["edge_factor"] << case["scale"]
    if family == "lattice":
        n = case["rows"] * case["cols"]
        return n, int(2 * 1.42 * n)
    if family == "batch":
        lo, hi = case["lo_log2"], case["hi_log2"]
        n = int(case["count"] * (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2)))
        return n, n * case["edge_factor"]
    return case["n"], case["m"]


def work(case):
    """Offsets and arcs read once (per superstep of PageRank, which needs them all again), weights
    where there are any, the result written once; one operation per arc and superstep (two for a
    rank's contribution and sum, one per mask bit of a source)."""
    n, m = _size(case)
    algo = case["algo"]
    if algo == "pagerank":
        steps = case["steps"]
        return {"bytes": steps * (4 * (n + 1) + 4 * m + 8 * n), "flops": 2 * m * steps}
    if algo == "mbfs":
        return {"bytes": 4 * (n + 1) + 4 * m + case["k"] * n, "flops": m * case["k"]}
    return {"bytes": 4 * (n + 1) + 4 * m * (2 if algo == "sssp" else 1) + 4 * n, "flops": m}


def exact(case, seed):
    """PageRank in 64 bits (the traversals return whole numbers).  The residual has no such value: it
    is the distance of two FP32 iterates, which near convergence is their rounding."""
    if case["algo"] != "pagerank":
        return None
    n, src, dst, _, starts = _arcs(case, seed)
    sizes = np.diff(starts)
    part = torch.repeat_interleave(torch.arange(len(sizes), device=DEV), torch.tensor(sizes, device=DEV))
    count = torch.tensor(sizes, device=DEV, dtype=torch.float64)
    outdeg = _out_degree(n, src)
    dangling = outdeg == 0
    d = float(np.float32(DAMPING))
    rank = (1.0 / count)[part]
    for _ in range(case["steps"]):
        gain = torch.zeros(n, dtype=torch.float64, device=DEV)
        gain.index_add_(0, dst, (rank / outdeg.clamp(min=1))[src])
        loose = torch.zeros(len(sizes), dtype=torch.float64, device=DEV)
        loose.index_add_(0, part[dangling], rank[dangling])
        rank = ((1.0 - d) / count + d * loose / count)[part] + d * gain
    return {"rank": rank, "residual": None}
