"""The calls whose speed counts, one case each.

A case is a graph and what a program does with it once it is loaded: a
traversal from a root, components, PageRank, the batched sources, a batch of
small graphs.  prepare() does what such a program does once (generate or read
the graph, load it, pick the schedule model or the PageRank shape, allocate
the page-locked host arrays that take the results), run() one query: the
application's initialisation, its loop, and the whole result on the host.

Graphs: R-MAT (a/b/c/d = .57/.19/.19/.05, hubs, the social and web graphs this
engine is benchmarked on), a road-like grid (thousands of levels, small
frontiers), uniformly random edges handed over unsorted (any vertex count,
no hubs), and disjoint unions of small R-MAT graphs of uneven size.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import wedge_amd as W

DAMPING = 0.85


def listed():
    return [
        # One query on a graph of a few thousand vertices, through the driver a
        # program calls first: launches, copies and allocations are all of it.
        {"name": "bfs_small", "app": "bfs_driver", "kind": "edges", "vertices": 3001, "degree": 11},
        # Hops from one vertex of a social graph under the learned schedule.
        {"name": "bfs_social", "app": "bfs", "kind": "rmat", "scale": 22, "ef": 16, "schedule": "learned"},
        # Hops over a road network: thousands of levels with small frontiers.
        {"name": "bfs_road", "app": "bfs", "kind": "grid", "rows": 1000, "cols": 1501, "schedule": "plain"},
        # Weighted distances on a social graph, FP64 weights.
        {"name": "sssp_social", "app": "sssp", "kind": "rmat", "scale": 21, "ef": 16, "schedule": "learned"},
        # Travel times over a road network, integer weights.
        {"name": "sssp_road", "app": "sssp", "kind": "grid", "rows": 700, "cols": 1001, "schedule": "plain"},
        # Components of an undirected social graph.
        {"name": "cc_social", "app": "cc", "kind": "rmat", "scale": 21, "ef": 16, "symmetric": True,
         "schedule": "plain"},
        # PageRank, FP64, shape tuned once per graph: the ordinary size ...
        {"name": "pr_mid", "app": "pr", "kind": "rmat", "scale": 20, "ef": 16, "iterations": 16, "fp32": False,
         "tune": True},
        # ... and a graph whose state is far larger than the caches, in the
        # binned shape that the tuner picks at such sizes.
        {"name": "pr_large", "app": "pr", "kind": "rmat", "scale": 24, "ef": 16, "iterations": 16, "fp32": False,
         "tune": False},
        # Hops from 64 vertices at once (closeness, landmark tables).
        {"name": "msbfs", "app": "msbfs", "kind": "rmat", "scale": 20, "ef": 23, "sources": 64},
        # Weighted distances from 64 vertices at once.
        {"name": "mssssp", "app": "mssssp", "kind": "rmat", "scale": 18, "ef": 16, "sources": 64},
        # Personalised PageRank of 32 users (recommendation).
        {"name": "ppr", "app": "ppr", "kind": "rmat", "scale": 20, "ef": 16, "sources": 32, "iterations": 16},
        # PageRank of many small graphs in one call.
        {"name": "batch_pr", "app": "batch_pr", "kind": "batch", "graphs": 64, "lo": 9, "hi": 15, "iterations": 16,
         "fp32": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    app = rng.choice(["bfs_driver", "bfs", "bfs", "sssp", "sssp", "cc", "pr", "pr", "msbfs", "mssssp", "ppr",
                      "batch_pr"])
    if app == "bfs_driver":
        return {"app": app, "kind": "edges", "vertices": _log_int(rng, 200, 60000), "degree": rng.randint(2, 40)}
    if app == "batch_pr":
        lo = rng.randint(8, 12)
        return {"app": app, "kind": "batch", "graphs": _log_int(rng, 8, 64), "lo": lo, "hi": lo + rng.randint(1, 3),
                "iterations": rng.randint(4, 24), "fp32": rng.random() < 0.5}
    if app in ("bfs", "sssp") and rng.random() < 0.4:
        return {"app": app, "kind": "grid", "rows": _log_int(rng, 60, 900), "cols": _log_int(rng, 60, 1100),
                "schedule": rng.choice(["plain", "learned"])}
    if app in ("bfs", "cc", "pr") and rng.random() < 0.3:
        case = {"app": app, "kind": "edges", "vertices": _log_int(rng, 5000, 1500000), "degree": rng.randint(3, 20)}
    else:
        top = {"bfs": 22, "sssp": 21, "cc": 20, "pr": 23, "msbfs": 20, "mssssp": 18, "ppr": 20}[app]
        case = {"app": app, "kind": "rmat", "scale": rng.randint(12, top), "ef": rng.randint(6, 18)}
    if app == "cc":
        case["symmetric"] = True
        if case["kind"] == "edges":
            case["degree"] = 1  # two edges per vertex: many components
    if app in ("bfs", "sssp", "cc"):
        case["schedule"] = rng.choice(["plain", "learned"])
    if app == "pr":
        case.update(iterations=rng.randint(4, 24), fp32=rng.random() < 0.5, tune=True)
    if app in ("msbfs", "mssssp"):
        case["sources"] = rng.randint(1, 64)
    if app == "ppr":
        case.update(sources=rng.randint(1, 32), iterations=rng.randint(4, 24))
    return case


# ---- inputs ------------------------------------------------------------------------


def _edges(case, seed):
    """Uniformly random edges in no order, without loops and repeats (both
    directions if the case asks for a symmetric graph)."""
    rng = np.random.default_rng(seed)
    v, n = case["vertices"], case["vertices"] * case["degree"]
    key = np.unique(rng.integers(0, v, n, dtype=np.int64) * v + rng.integers(0, v, n, dtype=np.int64))
    src, dst = key // v, key % v
    if case.get("symmetric"):
        key = np.unique(np.concatenate([src * v + dst, dst * v + src]))
        src, dst = key // v, key % v
    keep = np.nonzero(src != dst)[0]
    keep = keep[rng.permutation(keep.size)]
    return src[keep].astype(np.uint32), dst[keep].astype(np.uint32)


def _graph(case, seed):
    if case["kind"] == "grid":
        return W.grid(case["rows"], case["cols"], seed=seed)
    weighted = case["app"] in ("sssp", "mssssp")
    return W.rmat(case["scale"], case["ef"], seed=seed, symmetrize=bool(case.get("symmetric")),
                  weights="f64" if weighted else None)


def _members(case, seed):
    rng = np.random.default_rng([case["graphs"], case["lo"], case["hi"]])  # the sizes belong to the case
    scales = rng.integers(case["lo"], case["hi"] + 1, case["graphs"])
    efs = rng.integers(8, 33, case["graphs"])
    return [W.rmat(int(s), int(f), seed=seed + i) for i, (s, f) in enumerate(zip(scales, efs))]


def _sources(case, seed, od):
    """Roots or seeds: vertices with out-edges; on the grid the crossing with
    the most roads, which lies in the large component."""
    if case["kind"] == "grid":
        return np.array([int(np.argmax(od))], np.uint64)
    rng = np.random.default_rng(seed)
    return rng.choice(np.nonzero(od)[0], case.get("sources", 1), replace=False).astype(np.uint64)


def _out(shape, dtype):
    """Page-locked host array that a program keeps for its results."""
    return torch.empty(shape, dtype=dtype, pin_memory=True)


def prepare(case, seed):
    app = case["app"]
    ctx = W.Context(0)
    st = {"case": case, "ctx": ctx}
    if case["kind"] == "batch":
        ctx.load_batch(_members(case, seed))
        ctx.batch_autotune(case["iterations"], DAMPING, case["fp32"])
        st["out"] = _out(ctx.V, torch.float64)
    else:
        if case["kind"] == "edges":
            src, dst = _edges(case, seed)
            ctx.load_edges(case["vertices"], src, dst)
        else:
            ctx.load(_graph(case, seed))
            ctx.graph = None
        V = ctx.V
        if app not in ("cc", "pr"):
            st["roots"] = _sources(case, seed, ctx.outdegrees())
        if case.get("schedule") == "learned":
            W.mlp_load()
            ctx.set_schedule_model(W.mlp_get())
        if app == "pr":
            if case["tune"]:
                ctx.init_pr(DAMPING, case["fp32"])
                ctx.pr_autotune(2)
            else:
                ctx.set_pr_shape((8, 1, W.PR_BINNED))
        if app == "bfs":
            st["out"] = _out(V, torch.int64)
        elif app == "cc":
            st["out"] = _out(V, torch.int32)
        elif app == "sssp":
            st["out"] = _out(V, torch.int32 if case["kind"] == "grid" else torch.float64)
        elif app == "pr":
            st["out"] = _out(V, torch.float64)
        elif app in ("msbfs", "mssssp", "ppr"):
            st["out"] = _out((case["sources"], V), torch.int32 if app == "msbfs" else torch.float64)
    if "out" in st:
        st["ptr"] = [t.data_ptr() for t in (st["out"] if st["out"].dim() == 2 else st["out"].unsqueeze(0))]
    return st


# ---- one query ---------------------------------------------------------------------

_U64, _U32, _F64 = C.POINTER(C.c_uint64), C.POINTER(C.c_uint32), C.POINTER(C.c_double)


def _ok(rc):
    if rc != W.WG_OK:
        raise W.WedgeError(rc)


def run(st):
    case, ctx = st["case"], st["ctx"]
    app, lib, h = case["app"], ctx._lib, ctx.handle
    if app == "bfs_driver":
        packed, stats = ctx.run_bfs(int(st["roots"][0]))
        return [packed.view(np.int64), int(stats["vertices_reached"]), int(stats["edges_reached"])]
    ptr = st["ptr"]
    if app in ("bfs", "sssp", "cc"):
        sched = W.SCHEDULES[case["schedule"]]
        if app == "bfs":
            ctx.init_bfs(int(st["roots"][0]))
            ctx.converge(sched)
            _ok(lib.wg_read_bfs(h, C.cast(ptr[0], _U64)))
        elif app == "sssp":
            ctx.init_sssp(int(st["roots"][0]))
            ctx.converge(sched)
            _ok(lib.wg_read_sssp(h, ptr[0]))
        else:
            ctx.init_cc()
            ctx.converge(sched)
            _ok(lib.wg_read_cc(h, C.cast(ptr[0], _U32)))
    elif app == "pr":
        ctx.init_pr(DAMPING, case["fp32"])
        for _ in range(case["iterations"]):
            _ok(lib.wg_pr_iteration(h, None))
        _ok(lib.wg_read_ranks(h, C.cast(ptr[0], _F64)))
    elif app == "msbfs":
        levels, reached = ctx.msbfs(st["roots"])
        for s, p in enumerate(ptr):
            _ok(lib.wg_read_msbfs(h, s, C.cast(p, _U32)))
        return [st["out"], levels, reached]
    elif app == "mssssp":
        ctx.mssssp(st["roots"])
        for s, p in enumerate(ptr):
            _ok(lib.wg_read_mssssp(h, s, p))
    elif app == "ppr":
        ctx.ppr(st["roots"], case["iterations"], DAMPING)
        for s, p in enumerate(ptr):
            _ok(lib.wg_read_ppr(h, s, C.cast(p, _F64)))
    elif app == "batch_pr":
        ctx.batch_pr(case["iterations"], DAMPING, case["fp32"])
        _ok(lib.wg_read_batch_ranks(h, C.cast(ptr[0], _F64)))
    return st["out"]


# ---- what a pass cannot do without ---------------------------------------------------


def _size(case):
    """Vertices and (expected) edges of the case's graph."""
    kind = case["kind"]
    if kind == "grid":
        v = case["rows"] * case["cols"]
        return v, 2.5 * v
    if kind == "edges":
        v = case["vertices"]
        return v, v * case["degree"] * (2 if case.get("symmetric") else 1)
    if kind == "batch":
        v = case["graphs"] * sum(2.0 ** s for s in range(case["lo"], case["hi"] + 1)) / (case["hi"] - case["lo"] + 1)
        return v, 20 * v
    v = 1 << case["scale"]
    return v, v * case["ef"] * (2 if case.get("symmetric") else 1)


def work(case):
    """Traversals: the graph (offsets, sources, weights) read once, each
    vertex's result written once and copied out.  PageRank: per iteration the
    graph, the out-degrees and the contributions read and written (the batched
    one a row of FP32 contributions per vertex)."""
    v, e = _size(case)
    app = case["app"]
    if app in ("pr", "batch_pr"):
        c = 4 if case["fp32"] else 8
        return {"bytes": case["iterations"] * (4 * e + 8 * v + 2 * c * v) + 8 * v, "flops": case["iterations"] * e}
    if app == "ppr":
        n = case["sources"]
        return {"bytes": case["iterations"] * (4 * e + 8 * v + 8 * n * v) + 8 * n * v,
                "flops": case["iterations"] * e * n}
    n = case.get("sources", 1)
    value = {"bfs": 8, "bfs_driver": 8, "cc": 4, "msbfs": 4, "mssssp": 8,
             "sssp": 4 if case["kind"] == "grid" else 8}[app]
    weight = 0 if app not in ("sssp", "mssssp") else 4 if case["kind"] == "grid" else 8
    return {"bytes": 4 * (v + 1) + (4 + weight) * e + value * n * v, "flops": n * e if weight else 0}


def tolerance(case):
    """Hops, labels and distances are minima of the same values in any order:
    exact.  FP64 PageRank: sums of FP64 values in another order (1.4e-14 off
    64-bit sums in random order).  FP32-stored contributions: one rounding per
    contribution and iteration (2.6e-8; personalised 6.9e-9, where most of the
    mass stays at the seed)."""
    app = case["app"]
    if app in ("pr", "batch_pr"):
        return {"rel": 1.5e-7} if case["fp32"] else {"rel": 6e-14}
    if app == "ppr":
        return {"rel": 4e-8}
    return "exact"


# ---- the same in 64 bits, in plain torch ----------------------------------------------


def _csc(case, seed, dev):
    """Vertices, sources, destinations and weights; the edges in random order,
    so that a hub's sum does not meet itself in every neighbouring thread."""
    if case["kind"] == "edges":
        src, dst = _edges(case, seed)
        return case["vertices"], *(torch.from_numpy(a.astype(np.int64)).to(dev) for a in (src, dst)), None
    g = _graph(case, seed)
    src = torch.from_numpy(g.sources.astype(np.int64)).to(dev)
    deg = torch.from_numpy(np.diff(g.offsets.astype(np.int64))).to(dev)
    dst = torch.repeat_interleave(torch.arange(g.num_vertices, device=dev), deg)
    mix = torch.randperm(src.numel(), device=dev)
    w = None if g.weights is None else torch.from_numpy(g.weights.astype(np.float64)).to(dev)[mix]
    return g.num_vertices, src[mix], dst[mix], w


def _pagerank(v, src, dst, n, d, iterations):
    """n: the number of vertices of each vertex's graph; one[v]: that graph."""
    size, member, members = n
    od = torch.bincount(src, minlength=v).double()
    div = torch.where(od == 0, size, od)
    c = 1.0 / size / div
    for _ in range(iterations):
        acc = torch.zeros(v, dtype=torch.float64, device=src.device)
        for b in range(0, src.numel(), 1 << 26):
            acc.index_add_(0, dst[b:b + (1 << 26)], c[src[b:b + (1 << 26)]])
        s = torch.zeros(members, dtype=torch.float64, device=src.device).index_add_(0, member, acc)[member]
        c = ((acc + (1.0 - s) / size) * d + (1.0 - d) / size) / div
    return c * div


def exact(case, seed):
    app = case["app"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if app == "batch_pr":
        parts = []
        for g in _members(case, seed):
            v = g.num_vertices
            src = torch.from_numpy(g.sources.astype(np.int64)).to(dev)
            dst = torch.from_numpy(g.destinations().astype(np.int64)).to(dev)
            one = torch.full((v,), float(v), dtype=torch.float64, device=dev)
            parts.append(_pagerank(v, src, dst, (one, torch.zeros(v, dtype=torch.int64, device=dev), 1), DAMPING,
                                   case["iterations"]))
        return torch.cat(parts).cpu()
    if app == "pr":
        v, src, dst, _ = _csc(case, seed, dev)
        one = torch.full((v,), float(v), dtype=torch.float64, device=dev)
        return _pagerank(v, src, dst, (one, torch.zeros(v, dtype=torch.int64, device=dev), 1), DAMPING,
                         case["iterations"]).cpu()
    if app == "ppr":
        v, src, dst, _ = _csc(case, seed, dev)
        od = torch.bincount(src, minlength=v)
        seeds = torch.from_numpy(_sources(case, seed, od.cpu().numpy()).astype(np.int64)).to(dev)
        at = (seeds, torch.arange(len(seeds), device=dev))
        r = torch.zeros(v, len(seeds), dtype=torch.float64, device=dev)
        r[at] = 1.0
        for _ in range(case["iterations"]):
            c = torch.where(od[:, None] > 0, r / od.clamp(min=1).double()[:, None], torch.zeros_like(r))
            lost = r[od == 0].sum(0)
            acc = torch.zeros_like(r)
            for b in range(0, src.numel(), 1 << 22):
                acc.index_add_(0, dst[b:b + (1 << 22)], c[src[b:b + (1 << 22)]])
            acc[at] += lost
            r = acc * DAMPING
            r[at] += 1.0 - DAMPING
        return r.t().contiguous().cpu()
    if app in ("sssp", "mssssp") and case["kind"] == "rmat":
        v, src, dst, w = _csc(case, seed, dev)
        roots = _sources(case, seed, torch.bincount(src, minlength=v).cpu().numpy())
        rows = []
        for root in roots:
            dist = torch.full((v,), math.inf, dtype=torch.float64, device=dev)
            dist[int(root)] = 0.0
            while True:
                new = dist.clone().scatter_reduce_(0, dst, dist[src] + w, "amin")
                if torch.equal(new, dist):
                    break
                dist = new
            rows.append(dist)
        out = torch.stack(rows).cpu()
        return out if app == "mssssp" else out[0]
    return None
