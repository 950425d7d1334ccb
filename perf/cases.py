"""The workloads this engine's performance is measured on.

Each case is one call of a public search entry point on a resident graph, as a program
that keeps its graphs on the GPU makes it.  Graphs are the two families of the engine's
benchmark and tests: R-MAT power-law graphs (0.57, 0.19, 0.19, 0.05; edge factor 16;
self-loops and duplicates dropped, rows sorted; symmetrized or directed; n cut below
2^scale where a case asks for a ragged size) and 4-neighbour grids with 5% of the edges
deleted (meshes, road-like: thousands of levels).  They are generated on the GPU from the
seed and handed over as host CSR arrays, as a loader would.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  graph, sources, options and result buffers
    run(state)           one call; returns its whole result
    work(case)           bytes and operations of one call that no implementation avoids
    exact(case, seed)    PageRank results in 64 bits
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import mirrorofmapgraph_amd as mg

PAGERANK_ITERS = 50   # all-vertex Jacobi iterations of the PageRank benchmark
PPR_ITERS = 20        # the engine's default for personalized PageRank
BATCH_ROWS = 1 << 28  # largest sources x vertices of a drawn batched case


def listed() -> list[dict]:
    def rmat(n, algo, name, **kw):
        return dict({"name": name, "algo": algo, "graph": "rmat", "n": n, "symmetric": True, "relabel": False,
                     "wmax": 0, "k": 1, "host": False}, **kw)

    def grid(w, h, algo, name, **kw):
        return dict({"name": name, "algo": algo, "graph": "grid", "width": w, "height": h, "wmax": 0, "k": 1,
                     "host": False}, **kw)

    return [
        # the smallest interactive call: one BFS on a scale-16 graph through the Python
        # method, depths returned as a host array (latency and launches count)
        rmat(1 << 16, "bfs", "bfs_rmat16_host", host=True),
        # BFS on a large power-law graph kept with its degree-ordered copy: direction
        # optimisation, few wide levels
        rmat(1 << 21, "bfs", "bfs_rmat21", relabel=True),
        # BFS across a mesh: about 4,100 levels of at most a few thousand vertices
        grid(2048, 2048, "bfs", "bfs_grid2048"),
        # the headline weighted search: scale 22, weights 1..64, degree-ordered copy
        rmat(1 << 22, "sssp", "sssp_rmat22", relabel=True, wmax=64),
        # a directed graph of ragged size with an in-edge view, distances to a host array
        rmat(200_003, "sssp", "sssp_directed_host", symmetric=False, wmax=64, host=True),
        # weighted routing on a mesh with odd sides
        grid(1049, 999, "sssp", "sssp_grid1049x999", wmax=16),
        # component labelling of the large graph (the other half of the headline step)
        rmat(1 << 22, "cc", "cc_rmat22"),
        # PageRank on a directed graph, dangling vertices kept, 50 iterations
        rmat(1 << 21, "pagerank", "pagerank_rmat21", symmetric=False, relabel=True),
        # 256 BFS sources in one call (all-pairs samples, centrality estimates)
        rmat(1 << 20, "bfs_batch", "bfs_batch256_rmat20", relabel=True, k=256),
        # an odd number of weighted sources on a ragged graph without the renamed copy
        rmat(250_001, "sssp_batch", "sssp_batch100_rmat", wmax=64, k=100),
        # a cohort of personalized PageRank queries, the size serving starts one at
        rmat(1 << 20, "ppr_batch", "ppr_batch8_rmat20", relabel=True, k=8),
        # many weighted sources on a mesh
        grid(512, 512, "sssp_batch", "sssp_batch64_grid512", wmax=16, k=64),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    algo = rng.choice(["bfs", "bfs", "sssp", "sssp", "cc", "pagerank", "bfs_batch", "sssp_batch", "ppr_batch"])
    weighted = algo.startswith("sssp")
    if algo in ("bfs", "sssp", "cc", "bfs_batch", "sssp_batch") and rng.random() < 0.35:
        batched = algo.endswith("_batch")
        w = _log_int(rng, 100, 512 if batched else 1200)
        h = _log_int(rng, 100, 512 if batched else 1200)
        k = rng.randint(2, 64) if batched else 1
        return {"algo": algo, "graph": "grid", "width": w, "height": h, "wmax": 16 if weighted else 0, "k": k,
                "host": not batched and rng.random() < 0.3}
    if algo == "pagerank":
        n, k = _log_int(rng, 1 << 14, 1 << 21), 1
    elif algo == "ppr_batch":
        n, k = _log_int(rng, 1 << 14, 1 << 19), rng.randint(1, 32)
    elif algo == "bfs_batch":
        n = _log_int(rng, 1 << 14, 1 << 20)
        k = rng.randint(2, min(256, BATCH_ROWS // n))
    elif algo == "sssp_batch":
        n, k = _log_int(rng, 1 << 14, 250_000), rng.randint(2, 100)
    else:
        n, k = _log_int(rng, 1 << 14, 1 << 21), 1
    symmetric = rng.random() < (0.3 if algo == "pagerank" else 0.75)
    return {"algo": algo, "graph": "rmat", "n": n, "symmetric": symmetric, "relabel": rng.random() < 0.5,
            "wmax": rng.choice([16, 64, 255]) if weighted else 0, "k": k,
            "host": algo in ("bfs", "sssp", "cc") and n <= 1 << 18 and rng.random() < 0.4}


# ------------------------------------------------------------------ inputs
def _rmat_keys(n: int, symmetric: bool, gen: torch.Generator) -> torch.Tensor:
    """Sorted unique u * n + v of an R-MAT graph on ids below n."""
    scale = max(1, (n - 1).bit_length())
    m = 16 * n
    u = torch.zeros(m, dtype=torch.int32, device="cuda")
    v = torch.zeros(m, dtype=torch.int32, device="cuda")
    for _ in range(scale):
        r = torch.rand(m, device="cuda", generator=gen)
        down = r >= 0.76               # quadrants c and d
        right = ((r >= 0.57) & ~down) | (r >= 0.95)  # quadrants b and d
        u = 2 * u + down
        v = 2 * v + right
    ok = (u < n) & (v < n) & (u != v)
    u, v = u[ok].long(), v[ok].long()
    key = u * n + v
    if symmetric:
        key = torch.cat([key, v * n + u])
    return torch.unique(key)


def _grid_keys(w: int, h: int, gen: torch.Generator) -> torch.Tensor:
    """Sorted unique u * n + v of a symmetric 4-neighbour grid with 5% of its edges deleted."""
    n = w * h
    ids = torch.arange(n, device="cuda").view(h, w)
    a = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
    b = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
    kept = torch.rand(a.numel(), device="cuda", generator=gen) >= 0.05
    a, b = a[kept], b[kept]
    return torch.sort(torch.cat([a * n + b, b * n + a])).values


def _topology(case: dict, seed: int):
    """(n, row offsets, columns, weights or None, sources) as GPU tensors, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["graph"] == "grid":
        n = case["width"] * case["height"]
        key = _grid_keys(case["width"], case["height"], gen)
    else:
        n = case["n"]
        key = _rmat_keys(n, case["symmetric"], gen)
    u, v = key // n, key % n
    deg = torch.bincount(u, minlength=n)
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=off[1:])
    w = None
    if case["wmax"]:
        # the same weight in both directions of an undirected edge
        x = torch.minimum(u, v) * 0x9E3779B1 + torch.maximum(u, v) * 0x85EBCA77 + seed
        x = (x ^ (x >> 29)) * 0x2545F4914F6CDD1D
        w = (1 + ((x >> 33) & 0x7FFFFFFF) % case["wmax"]).int()
    alive = torch.nonzero(deg).reshape(-1)
    pick = torch.randint(0, alive.numel(), (case["k"],), device="cuda", generator=gen)
    return n, off.int(), v.int(), w, alive[pick]


def _is_symmetric(case: dict) -> bool:
    return case["graph"] == "grid" or case["symmetric"]


def prepare(case: dict, seed: int) -> dict:
    n, off, col, w, src = _topology(case, seed)
    host = mg.HostCSR(off.cpu().numpy(), col.cpu().numpy(), None if w is None else w.cpu().numpy())
    sym = _is_symmetric(case)
    graph = mg.Graph(host, symmetric=sym, build_csc=not sym, relabel=case.get("relabel", False))
    algo, k = case["algo"], case["k"]
    opt = {"out_on_device": 0 if case["host"] else 1}
    if algo == "pagerank":
        opt.update(pr_mode=mg.MG_PR_ALL, iter_num=PAGERANK_ITERS)
    state = {"algo": algo, "graph": graph, "opt": mg.options(**opt), "stats": mg.Stats(), "host": case["host"],
             "srcs": np.ascontiguousarray(src.cpu().numpy(), dtype=np.int32)}
    if not case["host"]:
        dtype = torch.float32 if algo in ("pagerank", "ppr_batch") else torch.int32
        shape = (k, n) if algo.endswith("_batch") else (n,)
        state["out"] = torch.empty(shape, dtype=dtype, device="cuda")
    return state


def run(state: dict):
    g, algo, opt, srcs = state["graph"], state["algo"], state["opt"], state["srcs"]
    if state["host"]:
        # the Python methods: results as host arrays
        return g.cc(opt) if algo == "cc" else getattr(g, algo)(int(srcs[0]), opt)
    # the C entry points: results left in the program's device buffer
    out = state["out"]
    args = [g.handle]
    if algo in ("bfs", "sssp"):
        args.append(int(srcs[0]))
    elif algo.endswith("_batch"):
        args += [srcs.ctypes.data_as(mg.I32P), len(srcs)]
    fn = getattr(mg.lib(), "mg_" + algo)
    mg.check(fn(*args, C.c_void_p(out.data_ptr()), C.byref(opt), C.byref(state["stats"])))
    return out


def work(case: dict) -> dict:
    """The topology (and weights) read once and the result written once; PageRank reads the
    topology every iteration.  Edge counts are the families' expected ones (R-MAT keeps about
    15.3 of 16 edges per vertex after deduplication)."""
    if case["graph"] == "grid":
        n = case["width"] * case["height"]
        m = 3.8 * n
    else:
        n = case["n"]
        m = (30.6 if case["symmetric"] else 15.5) * n
    k, algo = case["k"], case["algo"]
    topology = 4 * n + 4 * m
    if algo == "pagerank":
        return {"bytes": PAGERANK_ITERS * (topology + 12 * n), "flops": PAGERANK_ITERS * (m + 3 * n)}
    if algo == "ppr_batch":
        return {"bytes": PPR_ITERS * (topology + 8 * n * k), "flops": PPR_ITERS * k * (m + 3 * n)}
    weights = 4 * m if case["wmax"] else 0
    return {"bytes": topology + weights + 4 * n * k, "flops": 0}


def exact(case: dict, seed: int):
    algo = case["algo"]
    if algo not in ("pagerank", "ppr_batch"):
        return None
    n, off, col, _, src = _topology(case, seed)
    deg = (off[1:] - off[:-1]).double()
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), (off[1:] - off[:-1]).long())
    order = torch.argsort(col.long(), stable=True)  # in-edges grouped by target
    u, ends = row[order], torch.cumsum(torch.bincount(col.long(), minlength=n), 0)
    t = float(np.float32(0.15))
    damp = float(np.float32(1.0) - np.float32(0.15))

    def gather(x):
        c = torch.where(deg > 0, x / deg.clamp(min=1), torch.zeros_like(x))
        return torch.segment_reduce(c[u], "sum", offsets=torch.cat([ends.new_zeros(1), ends]), initial=0.0)

    if algo == "pagerank":
        x = torch.full((n,), t, dtype=torch.float64, device="cuda")
        for _ in range(PAGERANK_ITERS):
            x = t + damp * gather(x)
        return x.cpu()
    rows = []
    for s in src.tolist():
        x = torch.zeros(n, dtype=torch.float64, device="cuda")
        x[s] = 1.0
        for _ in range(PPR_ITERS):
            x = damp * gather(x)
            x[s] += t
        rows.append(x)
    return torch.stack(rows).cpu()
