"""Measured cases: the GAP kernels as a program calls them through gapbs_amd.gpu.

A case names an operation, the graph it runs on and its options.  prepare()
makes the graph's edge list on the GPU from the seed (R-MAT with the Graph500
parameters and permuted ids, uniform pairs, or a lattice with deletions and
shortcuts), builds the device graph and keeps what a program keeps between
calls: the handle, the roots, and page-locked result arrays where the entry
point takes one.  run() is one call with its results in host memory, the
reference's trial boundary (src/benchmark.h:107-109).
"""

import numpy as np
import torch

from gapbs_amd import gpu

DAMPING = 0.85
MAX_ITERS, EPSILON = 20, 1e-4  # the reference's PageRank defaults (src/pr.cc:98)


def listed():
    return [
        # One search of a small graph (Kronecker 16, the smallest named workload): launches and host latency.
        {"name": "bfs kron16", "op": "bfs", "graph": "kron", "n": 1 << 16, "degree": 16, "ordered": False},
        # One search of an ordinary graph, ids as uploaded.
        {"name": "bfs kron22", "op": "bfs", "graph": "kron", "n": 1 << 22, "degree": 16, "ordered": False},
        # The 64 searches of a benchmark run as one batched traversal, on the degree-ordered layout.
        {"name": "bfs64 kron20", "op": "bfs_batch", "graph": "kron", "n": 1 << 20, "degree": 16, "roots": 64, "ordered": True},
        # Shortest paths on a skewed graph with weights in [1, 255].
        {"name": "sssp kron22", "op": "sssp", "graph": "kron", "n": 1 << 22, "degree": 16, "delta": 16, "ordered": True},
        # Shortest paths on a road-like graph (long diameter, thousands of small steps, odd side).
        {"name": "sssp grid2047", "op": "sssp", "graph": "grid", "n": 2047 * 2047, "degree": 2, "delta": 1024, "ordered": False},
        # Sixteen shortest-path roots in one batched traversal.
        {"name": "sssp16 kron19", "op": "sssp_batch", "graph": "kron", "n": 1 << 19, "degree": 16, "roots": 16, "delta": 256, "ordered": True},
        # PageRank on the largest graph here, float scores.
        {"name": "pr kron24", "op": "pagerank", "graph": "kron", "n": 1 << 24, "degree": 16, "fp64": False, "ordered": True},
        # PageRank in double on a uniform graph of an odd size.
        {"name": "pr64 uniform3M", "op": "pagerank", "graph": "uniform", "n": 3000017, "degree": 16, "fp64": True, "ordered": False},
        # Connected components.
        {"name": "cc kron22", "op": "cc", "graph": "kron", "n": 1 << 22, "degree": 16, "ordered": False},
        # Betweenness from four roots, one after the other (the reference's -i4).
        {"name": "bc4 kron22", "op": "bc", "graph": "kron", "n": 1 << 22, "degree": 16, "roots": 4, "fp64": False, "ordered": True},
        # Betweenness from 64 roots in one batched traversal.
        {"name": "bc64 kron19", "op": "bc_batch", "graph": "kron", "n": 1 << 19, "degree": 16, "roots": 64, "fp64": False, "ordered": True},
        # Triangle counting with the degree relabelling that the reference times with it (src/tc.cc:97).
        {"name": "tc kron21", "op": "tc", "graph": "kron", "n": 1 << 21, "degree": 16, "ordered": False},
    ]


def _between(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["bfs", "bfs_batch", "sssp", "sssp_batch", "pagerank", "cc", "bc", "bc_batch", "tc"])
    top = {"bfs": 22, "bfs_batch": 19, "sssp": 22, "sssp_batch": 18, "pagerank": 23, "cc": 22, "bc": 21, "bc_batch": 18, "tc": 20}[op]
    n = _between(rng, 1 << 10, 1 << top)
    c = {"op": op, "graph": rng.choice(["kron", "kron", "uniform"]), "n": n, "degree": rng.choice([8, 12, 16]), "ordered": rng.random() < 0.5}
    if op in ("bfs", "sssp", "cc") and rng.random() < 0.25:
        side = _between(rng, 40, 2047)
        c.update(graph="grid", n=side * side, degree=2)
    if op in ("bfs", "sssp", "pagerank") and c["graph"] != "grid" and rng.random() < 0.2:
        c.update(directed=True, ordered=False)
    if op in ("bfs_batch", "bc_batch", "sssp_batch"):
        c["roots"] = rng.randint(4, 64) if op != "sssp_batch" else rng.randint(2, 16)
    if op == "bc":
        c["roots"] = rng.randint(1, 4)
    if op in ("sssp", "sssp_batch"):
        wide = c["graph"] == "grid" or op == "sssp_batch"
        c["delta"] = rng.choice([256, 512, 1024, 2048] if wide else [8, 16, 32, 64])
    if op in ("pagerank", "bc", "bc_batch"):
        c["fp64"] = rng.random() < 0.3
    if op == "tc":
        c["ordered"] = False
    return c


def _edges(case, seed):
    """The case's edge list on the GPU: (u, v, w or None), int32."""
    rng = torch.Generator(device="cuda").manual_seed(seed)
    n, weighted = case["n"], case["op"].startswith("sssp")
    if case["graph"] == "grid":
        side = int(round(n ** 0.5))
        at = torch.arange(side * side, dtype=torch.int32, device="cuda").view(side, side)
        u = torch.cat([at[:, :-1].reshape(-1), at[:-1].reshape(-1)])
        v = torch.cat([at[:, 1:].reshape(-1), at[1:].reshape(-1)])
        kept = torch.rand(u.numel(), device="cuda", generator=rng) >= 0.05
        extra = torch.randint(0, n, (2, u.numel() // 100), device="cuda", generator=rng, dtype=torch.int32)
        u, v = torch.cat([u[kept], extra[0]]), torch.cat([v[kept], extra[1]])
    elif case["graph"] == "uniform":
        u, v = torch.randint(0, n, (2, n * case["degree"]), device="cuda", generator=rng, dtype=torch.int32).unbind(0)
    else:  # R-MAT: A = 0.57, B = C = 0.19; ids scaled to [0, n) and permuted
        m, bits = n * case["degree"], max(1, (n - 1).bit_length())
        u = torch.zeros(m, dtype=torch.int32, device="cuda")
        v = torch.zeros(m, dtype=torch.int32, device="cuda")
        for _ in range(bits):
            r = torch.rand(m, device="cuda", generator=rng)
            u.mul_(2).add_(r > 0.76)
            v.mul_(2).add_(((r > 0.57) & (r <= 0.76)) | (r > 0.95))
        perm = torch.randperm(n, device="cuda", generator=rng).to(torch.int32)
        if n != 1 << bits:
            u, v = (x.to(torch.int64).mul_(n).bitwise_right_shift_(bits) for x in (u, v))
        u, v = perm[u], perm[v]
    u[0] = n - 1  # the builder counts vertices up to the largest id named
    w = None
    if weighted:
        top = 1000 if case["graph"] == "grid" else 255
        w = torch.randint(1, top + 1, (u.numel(),), device="cuda", generator=rng, dtype=torch.int32)
    return u, v, w


def _roots(case, seed, u, v):
    """Distinct end points of edges that are not loops: vertices a search can leave."""
    rng = torch.Generator(device="cuda").manual_seed(seed + 1)
    at = torch.randint(0, u.numel(), (4096,), device="cuda", generator=rng)
    ends = u[at][u[at] != v[at]].cpu().numpy()
    _, first = np.unique(ends, return_index=True)
    return np.ascontiguousarray(ends[np.sort(first)][: case.get("roots", 1)], dtype=np.int32)


def _host_array(shape, dtype):
    """A page-locked result array, as a program that reads results back on every call keeps."""
    return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()


def prepare(case, seed):
    u, v, w = _edges(case, seed)
    roots = _roots(case, seed, u, v)
    g, _ = gpu.build_graph(u.cpu().numpy(), v.cpu().numpy(), None if w is None else w.cpu().numpy(),
                           symmetrize=not case.get("directed", False), weighted=w is not None)
    if case["ordered"]:
        g.order_by_degree()
    op, n = case["op"], g.num_nodes
    out = None
    if op in ("bfs_batch", "sssp_batch"):
        out = _host_array((len(roots), n), torch.int32)
    elif op in ("sssp", "cc"):
        out = _host_array((n,), torch.int32)
    elif op in ("pagerank", "bc", "bc_batch"):
        out = _host_array((n,), torch.float32)
    return {"case": case, "graph": g, "roots": roots, "out": out}


def run(state):
    case, g, roots, out = state["case"], state["graph"], state["roots"], state["out"]
    op = case["op"]
    if op == "bfs":  # depths: parents are any valid tree, not one result
        return gpu.bfs(g, int(roots[0]), want_parent=False).depth
    if op == "bfs_batch":
        return gpu.bfs_batch(g, roots, out=out).depths
    if op == "sssp":
        return gpu.sssp(g, int(roots[0]), case["delta"], out=out).dist
    if op == "sssp_batch":
        return gpu.sssp_batch(g, roots, case["delta"], out=out).dist
    if op == "pagerank":
        return gpu.pagerank(g, MAX_ITERS, EPSILON, fp64=case["fp64"], out=out).scores
    if op == "cc":
        return gpu.cc(g, out=out).comp
    if op == "bc":
        return gpu.bc(g, roots, fp64=case["fp64"], out=out).scores
    if op == "bc_batch":
        return gpu.bc_batch(g, roots, fp64=case["fp64"], out=out).scores
    # tc: skewed graphs are relabelled first, as the reference's heuristic decides (src/tc.cc:75-100)
    if case["graph"] != "kron":
        return gpu.tc(g)[0]
    relabelled, _ = gpu.relabel_by_degree(g)
    return gpu.tc(relabelled)[0]


def work(case):
    """The graph read once and the result written once; list entries as drawn, before duplicates go."""
    n = case["n"]
    entries = n * case["degree"] * (1 if case.get("directed") else 2)
    read = 8 * (n + 1) + entries * (8 if case["op"].startswith("sssp") else 4)
    write = 8 if case["op"] == "tc" else 4 * n * (case["roots"] if case["op"] in ("bfs_batch", "sssp_batch") else 1)
    return {"bytes": read + write, "flops": 2 * entries if case["op"] in ("pagerank", "bc", "bc_batch") else 0}


def tolerance(case):
    # Four times the errors seen against exact(): scores are floats (half an
    # ulp, 3e-8, where the sums are exact or double); float dependencies and
    # score sums over a hub's successors are 5e-6 off.
    if case["op"] == "pagerank":
        return {"rel": 2e-7}
    if case["op"] in ("bc", "bc_batch"):
        return {"rel": 2e-7} if case["fp64"] else {"rel": 2e-5}
    return "exact"


def _lists(case, seed):
    """The squished graph's entries (source, destination), sorted by source, as int64 tensors."""
    u, v, _ = _edges(case, seed)
    n = int(max(u.max(), v.max())) + 1
    key = u.to(torch.int64) * n + v
    if not case.get("directed", False):
        key = torch.cat([key, v.to(torch.int64) * n + u])
    key = torch.unique(key)
    src, dst = key // n, key % n
    kept = src != dst
    return n, src[kept], dst[kept]


def _sums(values, at, n):
    return torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, at, values)


def exact(case, seed):
    if case["op"] not in ("pagerank", "bc", "bc_batch"):
        return None  # whole numbers
    n, src, dst = _lists(case, seed)
    if case["op"] == "pagerank":
        degree = _sums(torch.ones_like(src, dtype=torch.float64), src, n).clamp_(min=1)
        score = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
        for _ in range(MAX_ITERS):
            new = (1 - DAMPING) / n + DAMPING * _sums((score / degree)[src], dst, n)
            change = float((new - score).abs().sum())
            score = new
            if change < EPSILON:
                break
        return score.cpu().numpy()
    u, v, _ = _edges(case, seed)
    total = torch.zeros(n, dtype=torch.float64, device="cuda")
    for root in _roots(case, seed, u, v).tolist():
        depth = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        paths = torch.zeros(n, dtype=torch.float64, device="cuda")
        depth[root], paths[root] = 0, 1
        levels, level = [], 0
        while True:
            e = torch.nonzero((depth[src] == level) & (depth[dst] < 0)).view(-1)
            if e.numel() == 0:
                break
            a, b = src[e], dst[e]
            depth[b] = level + 1
            paths += _sums(paths[a], b, n)
            levels.append((a, b))
            level += 1
        delta = torch.zeros(n, dtype=torch.float64, device="cuda")
        for a, b in reversed(levels):
            delta += _sums(paths[a] / paths[b] * (1 + delta[b]), a, n)
        total += delta
    return (total / total.max()).cpu().numpy()
