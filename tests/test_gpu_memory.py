"""Traversals and batched queries where device memory ends: what a context can do
without (the vertex records of the one-workgroup levels on graphs of few edges
per vertex, the stage that results pass through) gives way to what a call needs.

Each case runs in a process of its own, in which hipMalloc comes from a small
library that refuses what exceeds a limit; the limits are sized from the same
calls without one."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

LIMITER = r"""
#include <stddef.h>
static struct { void* p; size_t n; } held[4096];
static size_t used, peak, limit = ~(size_t)0, refused;
static int (*real_malloc)(void**, size_t), (*real_free)(void*);
void limiter_real(void* m, void* f) { real_malloc = (int (*)(void**, size_t))m; real_free = (int (*)(void*))f; }
void limiter_set(size_t n) { limit = n; }
size_t limiter_used(void) { return used; }
size_t limiter_refused(void) { return refused; }
size_t limiter_peak(void) { size_t p = peak; peak = used; return p; }
int hipMalloc(void** p, size_t n)
{
    if (used + n > limit) {
        ++refused;
        return 2; /* hipErrorOutOfMemory */
    }
    int e = real_malloc(p, n);
    for (int i = 0; !e && i < 4096; ++i)
        if (!held[i].p) {
            held[i].p = *p;
            held[i].n = n;
            used += n;
            peak = used > peak ? used : peak;
            break;
        }
    return e;
}
int hipFree(void* p)
{
    for (int i = 0; p && i < 4096; ++i)
        if (held[i].p == p) {
            used -= held[i].n;
            held[i].p = NULL;
        }
    return real_free(p);
}
"""

CHILD = r"""
import ctypes, sys
lim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in ("limiter_used", "limiter_refused", "limiter_peak"):
    getattr(lim, f).restype = ctypes.c_size_t
import numpy as np
import wedge_amd as W
W.host_threads()  # loads the libraries, and with them the runtime
hip = ctypes.CDLL("libamdhip64.so.7")
lim.limiter_real(ctypes.cast(hip.hipMalloc, ctypes.c_void_p), ctypes.cast(hip.hipFree, ctypes.c_void_p))
NONE = ctypes.c_size_t(2**64 - 1)


def limit(n):
    lim.limiter_set(NONE if n is None else ctypes.c_size_t(n))


case = sys.argv[2]
app = "sssp" if case == "sssp" else "bfs"
g = W.grid(150, 170, seed=5)
V = g.num_vertices
records = 64 * V + 8 * 2**20 if app == "sssp" else 32 * V
root = g.max_outdegree_vertex()


def query(c):
    (c.init_sssp if app == "sssp" else c.init_bfs)(root)
    c.converge(W.SCHED_FRONTIER)
    return c.read_sssp() if app == "sssp" else c.read_bfs()


def refused(f):
    try:
        f()
    except W.WedgeError as e:
        return e.code
    return W.WG_OK


c = W.Context(0, relabel=True)
c.load(g)
assert lim.limiter_used() > 0, "hipMalloc is not the limiter's"
lim.limiter_peak()
want = query(c)
need = lim.limiter_peak()
if case == "batched":
    # a BFS leaves its records and the results' stage; the batched buffers get their room
    roots = np.arange(64, dtype=np.uint64)
    base = lim.limiter_used()
    c.msbfs(roots)
    extra = lim.limiter_peak() - base
    want64 = c.read_msbfs(9)
c.close()

if case == "batched":
    for short in (1, records // 2, records):
        c = W.Context(0, relabel=True)
        c.load(g)
        query(c)
        limit(lim.limiter_used() + extra - short)
        c.msbfs(roots)
        assert np.array_equal(c.read_msbfs(9), want64), short
        assert np.array_equal(query(c), want), short
        limit(None)
        c.close()
else:
    for short in (1, 4096, records // 2, records):
        c = W.Context(0, relabel=True)
        c.load(g)
        limit(need - short)
        assert np.array_equal(query(c), want), short
        n = lim.limiter_refused()
        assert np.array_equal(query(c), want), short
        assert lim.limiter_refused() == n, "what there was no room for is tried again"
        limit(None)
        c.close()
    # less than the traversal needs: an error, nothing to go on from, and a fresh start
    # once there is room
    c = W.Context(0, relabel=True)
    c.load(g)
    limit(lim.limiter_used() + 4 * V)
    assert refused(lambda: query(c)) in (W.WG_E_HIP, W.WG_E_NOMEM)
    assert refused(lambda: c.converge(W.SCHED_FRONTIER)) == W.WG_E_STATE
    limit(None)
    assert np.array_equal(query(c), want)
    c.close()
assert lim.limiter_used() == 0
print("ok")
"""


@pytest.fixture(scope="module")
def limiter(tmp_path_factory):
    d = tmp_path_factory.mktemp("limiter")
    src, lib = d / "limiter.c", d / "limiter.so"
    src.write_text(LIMITER)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(lib), str(src)], check=True)
    return str(lib)


@pytest.mark.parametrize("case", ["bfs", "sssp", "batched"])
def test_optional_memory_gives_way(limiter, case):
    r = subprocess.run([sys.executable, "-c", CHILD, limiter, case], cwd=ROOT, capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
