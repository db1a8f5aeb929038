"""The branches that a graph's size selects, each at a size that takes it:
pull bins of 4K, 8K and 16K vertices of the binned layout, the 128-edge tiles of
the 64-source SSSP with and without marked destinations (hub lists cut into
chunks; the 512-edge tiles of larger graphs are tests/test_gpu_configs.py's 64
sources on rmat-s24), one to eight wavefronts per tile of the personalised
PageRank, BFS levels and SSSP rounds in one workgroup (long out-lists cut into
chunks, levels handed back and forth, the pulls of a capped SSSP), traversals
from few and many roots, and results stored to page-locked memory by the kernel
or copied.  Against the oracle: exact for BFS, CC and SSSP, 1e-10 L1 for FP64
PageRank (sums of FP64 values in another order), 2e-7 L1 for FP32-stored
contributions (one rounding of 6e-8 per contribution)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import wedge_amd as W

pytestmark = pytest.mark.gpu


def _sparse(V, n, seed, symmetric=False, weights=None):
    """n random edges over V vertices, some into and out of a hub, some among
    the last vertices (the last window and bin)."""
    rng = np.random.default_rng(seed)
    src = np.concatenate([rng.integers(0, V, n), rng.integers(0, V, 3000), np.full(3000, 7),
                          rng.integers(V - 50, V, 300)])
    dst = np.concatenate([rng.integers(0, V, n), np.full(3000, 7), rng.integers(0, V, 3000),
                          rng.integers(V - 50, V, 300)])
    if symmetric:
        src, dst = np.concatenate([src, dst]), np.concatenate([dst, src])
    w = None
    if weights == "f64":
        w = rng.random(src.size) + 1e-3
    elif weights == "int":
        w = rng.integers(1, 1000, src.size).astype(np.uint32)
    return W.from_edges(V, src, dst, w, dedup=True)


# 1024 bins of 4K, 8K and 16K vertices are the smallest counts that select them
@pytest.mark.parametrize("V", [(1 << 22) - 1, 1 << 23, (1 << 24) + 5])
def test_binned_bin_sizes(V):
    g = _sparse(V, 40000, 3)
    gs = _sparse(V, 20000, 4, symmetric=True)
    c = W.Context(0, relabel=False)
    try:
        c.load(g)
        ref, _ = oracle.Oracle.of(g, 8).pr(4, 0.85)
        for fp32 in (False, True):
            c.set_pr_shape((8, 1, W.PR_BINNED))
            ranks, _ = c.run_pr(iterations=4, damping=0.85, contrib_fp32=int(fp32))
            assert float(np.abs(ranks - ref).sum()) <= (2e-7 if fp32 else 1e-10), fp32
        c.set_option(W.OPT_MS_BINNED, 1)
        roots = np.array([7, V - 3, 7], np.uint64)
        c.msbfs(roots, schedule="dense")
        for i, r in enumerate(roots):
            assert np.array_equal(c.read_msbfs(i), oracle.Oracle.of(g, 8).bfs(int(r))[1]), i
        c.set_option(W.OPT_MIN_BINNED, 1)
        c.load(gs)
        labels, _ = c.run_cc(schedule="dense")
        assert np.array_equal(labels.astype(np.float64), oracle.Oracle.of(gs, 8).cc()[0])
    finally:
        c.close()


@pytest.mark.parametrize("weights", ["f64", "int"])
@pytest.mark.parametrize("relabel", [False, True])
def test_mssssp_hub_lists(weights, relabel):
    """A hub with 3000 out-edges (three chunks of the marking) and 3000 in-edges
    (several heavy tiles), every schedule."""
    g = _sparse(5003, 30000, 5, weights=weights)
    orc = oracle.Oracle.of(g, 8)
    roots = np.concatenate([[7, 5002], np.arange(11)]).astype(np.uint64)
    want = [orc.sssp(int(r))[0] for r in roots]
    c = W.Context(0, relabel=relabel)
    try:
        c.load(g)
        for schedule in ("plain", "dense", "frontier"):
            c.mssssp(roots, schedule=schedule)
            for i in range(len(roots)):
                got = c.read_mssssp(i)
                if weights == "int":  # the oracle's unreached is UINT64_MAX
                    got = np.where(got == np.uint32(0xFFFFFFFF), np.uint64(2**64 - 1), got.astype(np.uint64))
                assert np.array_equal(got, want[i]), (schedule, i)
    finally:
        c.close()


# tiles of at most 256 destinations: 4, 79, 1563 and 7813 of them give 8, 8, 4
# and 1 wavefronts per tile on 256 CUs
@pytest.mark.parametrize("V", [1000, 20000, 400001, 2000000])
def test_ppr_wavefronts_per_tile(V):
    g = _sparse(V, 2 * V, 6)
    seeds = np.array([7, V - 2, 0, 3], np.uint64)
    want = oracle.Oracle.of(g, 8).ppr(seeds, 5, 0.85)
    c = W.Context(0)
    try:
        c.load(g)
        c.ppr(seeds, 5, 0.85)
        for i in range(len(seeds)):
            assert float(np.abs(c.read_ppr(i) - want[i]).sum()) <= 2e-7, i
    finally:
        c.close()


def _levels_graph(name):
    """Road-like graphs (at most 4 out-edges per vertex) whose levels take each
    road through the one-workgroup levels."""
    if name == "grid":  # levels stay small
        return W.grid(37, 53, seed=4, p_keep=0.9)
    if name == "wide":  # levels outgrow one workgroup (2048 vertices) and shrink again
        return _broom(5000)
    return _broom(300)


def _broom(width):
    """A path, a fan of `width` vertices (more destinations than a record
    holds) each with a chain of 5, all chains meeting in one vertex, and a path."""
    n = 0
    src, dst = [], []

    def chain(a, length):
        nonlocal n
        for _ in range(length):
            src.append(a)
            dst.append(n)
            a = n
            n += 1
        return a

    n = 1
    hub = chain(0, 20)
    ends = [chain(hub, 6) for _ in range(width)]
    meet = n
    n += 1
    for e in ends:
        src.append(e)
        dst.append(meet)
    chain(meet, 30)
    return W.from_edges(n, src, dst)


@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("name", ["grid", "wide", "fan"])
def test_bfs_levels_in_one_workgroup(name, relabel):
    g = _levels_graph(name)
    root = 0 if name != "grid" else g.max_outdegree_vertex()
    _, depth, _ = oracle.Oracle.of(g, 4).bfs(root)
    W.mlp_load()
    c = W.Context(0, relabel=relabel)
    try:
        c.load(g)
        c.set_schedule_model(W.mlp_get())
        for schedule, cap in ((W.SCHED_FRONTIER, 0), (W.SCHED_PLAIN, 0), (W.SCHED_LEARNED, 0), (W.SCHED_FRONTIER, 9)):
            got = []
            for wgs in (0, 32, 1):
                c.set_fused_levels(wgs)
                c.init_bfs(root)
                it = c.converge(schedule, max_iterations=cap)
                got.append((c.read_bfs(), it))
                if schedule == W.SCHED_FRONTIER and wgs == 32:
                    assert c.fused_level_count() > 0
                if cap:  # what follows finds visited, frontier and depths as after any level
                    c.edge_pull(W.APP_BFS, W.MODE_DENSE)
                    got[-1] += (c.read_bfs(),)
            for other in got[1:]:
                assert other[1] == got[0][1], (schedule, cap)
                for a, b in zip(got[0][::2], other[::2]):
                    assert np.array_equal(a, b), (schedule, cap)
            if not cap:
                assert np.array_equal(W.bfs_depth(got[0][0]), depth), schedule
    finally:
        c.close()


def _weighted(g, kind, seed):
    """g with weights: random, all equal (ties everywhere), or many zeros."""
    rng = np.random.default_rng(seed)
    E = g.num_edges
    w = {"random": rng.integers(1, 1000, E), "equal": np.full(E, 7), "zeros": rng.integers(0, 3, E)}[kind]
    return w.astype(np.uint32), w.astype(np.float64) * 0.37


# at most 4 out-edges per vertex: a grid; a fan of 300 and one of 20000 (more
# than the near queue holds); random edges (more vertices waiting than one
# workgroup keeps)
@pytest.mark.parametrize("kind", ["random", "equal", "zeros"])
@pytest.mark.parametrize("graph", ["grid", "fan", "wide", "random"])
def test_sssp_rounds_in_one_workgroup(graph, kind):
    g = {"grid": lambda: W.grid(61, 83, seed=4), "fan": lambda: _broom(300), "wide": lambda: _broom(20000),
         "random": lambda: _sparse(200000, 500000, 8)}[graph]()
    root = 7 if graph == "random" else 0
    if graph == "grid":
        root = g.max_outdegree_vertex()
    for w in _weighted(g, kind, 5):
        gw = W.Graph(g.offsets, g.sources, w)
        want = oracle.Oracle.of(gw, 8).sssp(root)[0]
        c = W.Context(0)
        try:
            c.load(gw)
            for schedule in (W.SCHED_FRONTIER, W.SCHED_PLAIN):
                c.init_sssp(root)
                it, _ = c.converge(schedule)
                got = c.read_sssp()
                if w.dtype == np.uint32:
                    got = np.where(got == np.uint32(0xFFFFFFFF), np.uint64(2**64 - 1), got.astype(np.uint64))
                assert np.array_equal(got, want), (w.dtype, schedule)
                assert c.validate() == 0 or kind == "zeros"
                c.init_sssp(root)  # stopped early
                assert c.converge(schedule, max_iterations=3)[0] == 3
                c.set_fused_levels(0, (W.APP_SSSP,))  # the same without these rounds
                c.init_sssp(root)
                c.converge(schedule)
                again = c.read_sssp()
                if w.dtype == np.uint32:
                    again = np.where(again == np.uint32(0xFFFFFFFF), np.uint64(2**64 - 1), again.astype(np.uint64))
                assert np.array_equal(again, want), (w.dtype, schedule)
                c.close()
                c = W.Context(0)
                c.load(gw)
        finally:
            c.close()


def _hubs(degrees):
    """Vertices with the given out-degrees one after another, two levels apart:
    each leads to leaves of its own, the first of them to the next vertex."""
    src, dst, n = [], [], 1
    hub = 0
    for d in degrees:
        src.append(np.full(d, hub))
        dst.append(np.arange(n, n + d))
        src.append(np.array([n]))
        dst.append(np.array([n + d]))
        hub = n + d
        n += d + 1
    return W.from_edges(n, np.concatenate(src), np.concatenate(dst))


def _many_lists(mids, degree, leaves):
    """A root to `mids` vertices, each with `degree` random ones of `leaves`."""
    rng = np.random.default_rng(9)
    src = np.concatenate([np.zeros(mids, np.int64), np.repeat(np.arange(1, mids + 1), degree)])
    dst = np.concatenate([np.arange(1, mids + 1), mids + 1 + rng.integers(0, leaves, mids * degree)])
    return W.from_edges(mids + 1 + leaves, src, dst, dedup=True)


# out-lists longer than a vertex's record: up to one chunk of 256 out-edges, one
# more, several rounds of the 16 wavefronts, and for SSSP the longest that one
# workgroup takes (65536) and one more
@pytest.mark.parametrize("relabel", [False, True])
def test_bfs_long_lists_in_one_workgroup(relabel):
    g = _hubs([1, 7, 8, 9, 255, 256, 257, 511, 512, 513, 3000, 12287, 12288, 12289, 20])
    _, depth, _ = oracle.Oracle.of(g, 4).bfs(0)
    c = W.Context(0, relabel=relabel)
    try:
        c.load(g)
        for schedule in (W.SCHED_FRONTIER, W.SCHED_PLAIN):
            got = []
            for wgs in (0, 32):
                c.set_fused_levels(wgs)
                c.init_bfs(0)
                got.append((c.converge(schedule), c.read_bfs()))
            assert got[0][0] == got[1][0], schedule
            assert np.array_equal(got[0][1], got[1][1]), schedule
            assert np.array_equal(W.bfs_depth(got[1][1]), depth), schedule
    finally:
        c.close()


def test_bfs_small_levels_between_wide_ones():
    """Fans of 3000 (more than one workgroup takes) with chains between them, short
    of what a fused run waits for before it hands levels back, just that, and
    several times as long: the run and the workgroup take turns."""
    src, dst, n, at = [], [], 1, 0
    for length in (1, 3, 7, 8, 9, 16, 17, 70, 8, 9, 40, 1):
        src.append(np.full(3000, at))
        dst.append(np.arange(n, n + 3000))
        chain = np.concatenate([[n], np.arange(n + 3000, n + 3000 + length)])
        src.append(chain[:-1])
        dst.append(chain[1:])
        n += 3000 + length
        at = n - 1
    g = W.from_edges(n, np.concatenate(src), np.concatenate(dst))
    _, depth, _ = oracle.Oracle.of(g, 4).bfs(0)
    c = W.Context(0)
    try:
        c.load(g)
        got = []
        for wgs in (0, 32, 2):
            c.set_fused_levels(wgs)
            c.init_bfs(0)
            got.append((c.converge(W.SCHED_FRONTIER), c.read_bfs()))
        for it, packed in got:
            assert it == got[0][0]
            assert np.array_equal(packed, got[0][1])
            assert np.array_equal(W.bfs_depth(packed), depth)
    finally:
        c.close()


# many: 3000 vertices at one distance (equal weights), a chunk each, where a
# round holds 2048
@pytest.mark.parametrize("graph", ["hubs", "many"])
def test_sssp_long_lists_in_one_workgroup(graph):
    g = _hubs([1, 5, 6, 7, 8, 255, 256, 257, 513, 4097, 65536, 65537, 20]) if graph == "hubs" else \
        _many_lists(3000, 9, 20000)
    assert g.num_edges <= 4 * g.num_vertices
    for kind in ("equal", "random"):
        for w in _weighted(g, kind, 11):
            gw = W.Graph(g.offsets, g.sources, w)
            want = oracle.Oracle.of(gw, 8).sssp(0)[0]
            if w.dtype == np.uint32:
                want = np.where(want == np.uint64(2**64 - 1), np.uint64(0xFFFFFFFF), want).astype(np.uint32)
            c = W.Context(0)
            try:
                c.load(gw)
                its = []
                for rounds in (True, False):
                    if not rounds:
                        c.set_fused_levels(0, (W.APP_SSSP,))
                    c.init_sssp(0)
                    its.append(c.converge(W.SCHED_FRONTIER)[0])
                    assert np.array_equal(c.read_sssp(), want), (kind, w.dtype, rounds)
                if graph == "hubs" and kind == "random":  # nearest first takes more, smaller rounds
                    assert its[0] > its[1], its
            finally:
                c.close()


def _hop_distances(g, w, root, k):
    """Shortest distances over paths of at most k edges (unreached: infinite)."""
    d = np.full(g.num_vertices, np.inf)
    d[root] = 0.0
    dst = g.destinations()
    for _ in range(k):
        new = d.copy()
        np.minimum.at(new, dst, d[g.sources] + w)
        d = new
    return d


# at most 4 out-edges per vertex, where a loop without a cap takes nearest-first
# rounds; integer weights below 2^32 and their sums are exact in FP64
@pytest.mark.parametrize("graph", ["grid", "fan"])
@pytest.mark.parametrize("cap", [1, 3, 24])
def test_sssp_after_capped_pulls(graph, cap):
    g = W.grid(61, 83, seed=4) if graph == "grid" else _broom(300)
    root = g.max_outdegree_vertex() if graph == "grid" else 0
    for w in _weighted(g, "random", 6):
        bound = _hop_distances(g, w.astype(np.float64), root, cap)
        gw = W.Graph(g.offsets, g.sources, w)
        best = oracle.Oracle.of(gw, 8).sssp(root)[0]
        c = W.Context(0)
        try:
            c.load(gw)
            for schedule in (W.SCHED_FRONTIER, W.SCHED_PLAIN, W.SCHED_DENSE):
                c.init_sssp(root)
                assert c.converge(schedule, max_iterations=cap)[0] <= cap
                got = c.read_sssp()
                if w.dtype == np.uint32:
                    best_f = np.where(best == np.uint64(2**64 - 1), np.inf, best.astype(np.float64))
                    got = np.where(got == np.uint32(0xFFFFFFFF), np.inf, got.astype(np.float64))
                else:
                    best_f = best
                assert (got <= bound).all(), (w.dtype, schedule)
                assert (got >= best_f).all(), (w.dtype, schedule)
        finally:
            c.close()


# up to 4096 roots have offsets for a push of their out-edges, more only a total
@pytest.mark.parametrize("n", [2, 4095, 4096, 4097, 9001])
def test_many_roots(n):
    g = _sparse(20011, 70000, 12, weights="int")
    roots = np.random.default_rng(n).choice(20011, n, replace=False).astype(np.uint64)
    total = int(g.outdegrees()[roots.astype(np.int64)].sum())
    dst = g.destinations()

    def fixpoint(d, w):
        while True:
            new = d.copy()
            np.minimum.at(new, dst, d[g.sources] + w)
            if np.array_equal(new, d):
                return d
            d = new

    start = np.full(g.num_vertices, np.inf)
    start[roots.astype(np.int64)] = 0.0
    c = W.Context(0)
    try:
        c.load(g)
        for init, read, w in ((c.init_bfs_roots, lambda: W.bfs_depth(c.read_bfs()), 1.0),
                              (c.init_sssp_roots, c.read_sssp, g.weights.astype(np.float64))):
            want = fixpoint(start, w)
            for schedule in (W.SCHED_PLAIN, W.SCHED_FRONTIER):
                init(roots)
                c.converge(schedule)
                got = read()
                assert np.array_equal(np.where(got == np.uint32(0xFFFFFFFF), np.inf, got.astype(np.float64)), want)
            # the roots' out-degrees choose the first pull
            pct = total * 100 // g.num_edges
            for threshold, frontier in ((pct, g.num_edges * pct // 100 >= total), (pct + 1, True)):
                init(roots)
                assert c.converge(W.SCHED_PLAIN, threshold_pct=threshold, max_iterations=1) == (1, int(frontier))
    finally:
        c.close()


# page-locked memory: at an allocation's start, inside one, ending with one, at
# no multiple of the element size (copied), and over 32 MiB (copied); the
# elements around the result keep their value
@pytest.mark.parametrize("V", [1, 65, 70001, (1 << 22) + 3])
@pytest.mark.parametrize("relabel", [False, True])
def test_results_in_page_locked_memory(V, relabel):
    import ctypes

    rng = np.random.default_rng(V)
    n = min(2 * V, 200000)
    g = W.from_edges(V, rng.integers(0, V, n), rng.integers(0, V, n), rng.integers(1, 9, n).astype(np.uint32))
    c = W.Context(0, relabel=relabel)
    lib, h = c._lib, c.handle

    def check(read, want):
        want = np.ascontiguousarray(want)
        for before, after in ((0, 64), (64, 0), (want.itemsize, want.itemsize), (want.itemsize // 2 + 1, 64)):
            size = before + want.nbytes + after
            mem = ctypes.c_void_p()
            assert lib.hipHostMalloc(ctypes.byref(mem), ctypes.c_size_t(size), ctypes.c_uint(0)) == 0
            try:
                b = np.ctypeslib.as_array(ctypes.cast(mem, ctypes.POINTER(ctypes.c_uint8)), (size,))
                b[:] = 0x5A
                assert read(ctypes.c_void_p(mem.value + before)) == 0
                assert b[before:before + want.nbytes].tobytes() == want.tobytes(), (before, after)
                assert (b[:before] == 0x5A).all() and (b[before + want.nbytes:] == 0x5A).all()
            finally:
                assert lib.hipHostFree(mem) == 0

    def as_(t, f, *a):
        return lambda p: f(h, *a, ctypes.cast(p, ctypes.POINTER(t)))

    try:
        c.load(g)
        c.init_bfs(0)
        c.converge(W.SCHED_FRONTIER)
        check(as_(ctypes.c_uint64, lib.wg_read_bfs), c.read_bfs())
        c.init_sssp(0)
        c.converge(W.SCHED_FRONTIER)
        check(lambda p: lib.wg_read_sssp(h, p), c.read_sssp())
        ranks, _ = c.run_pr(iterations=2)
        check(as_(ctypes.c_double, lib.wg_read_ranks), ranks)
        if V > 1 << 20:
            return
        roots = np.array([0, V - 1], np.uint64)
        c.msbfs(roots)
        check(as_(ctypes.c_uint32, lib.wg_read_msbfs, 1), c.read_msbfs(1))
        c.mssssp(roots)
        check(lambda p: lib.wg_read_mssssp(h, 1, p), c.read_mssssp(1))
        c.ppr(roots, 2, 0.85)
        check(as_(ctypes.c_double, lib.wg_read_ppr, 1), c.read_ppr(1))
    finally:
        c.close()
