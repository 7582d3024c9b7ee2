"""Device allocations that fail, and pinned ones that are given back. A copy of the library is loaded behind a stand-in
for hipMalloc that fails when told to (the device itself is never filled): a rebuild that runs out of memory, at whichever of its allocations, leaves no
tree that a search could walk, and the next build works; counts whose tight boxes find no room do without them."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
long shim_calls = 0, shim_allow = -1;  /* allocations so far; how many succeed from now on (-1: all) */
long shim_pinned = 0;                  /* pinned allocations that live */
static void *hip(const char *name) { return dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), name); }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    int e = ((int (*)(void **, size_t, unsigned))hip("hipHostMalloc"))(p, n, flags);
    if (!e) shim_pinned++;
    return e;
}
int hipHostFree(void *p) {
    int e = ((int (*)(void *))hip("hipHostFree"))(p);
    if (!e && p) shim_pinned--;
    return e;
}
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t) = 0;
    if (!real) real = (int (*)(void **, size_t))hip("hipMalloc");
    shim_calls++;
    if (shim_allow == 0) return 2; /* hipErrorOutOfMemory */
    if (shim_allow > 0) shim_allow--;
    return real(p, n);
}
"""


class Shim:
    def __init__(self, path):
        self.h = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self._calls, self._allow, self._pinned = (C.c_long.in_dll(self.h, f"shim_{n}") for n in ("calls", "allow", "pinned"))

    def allow(self, n):
        self._allow.value = n

    def calls(self):
        return self._calls.value

    def pinned(self):
        return self._pinned.value


def context(path):
    """A context of the library at `path`."""
    keep = A.lib(), A.LIB_PATH
    A._LIB, A.LIB_PATH = None, path
    try:
        return A.Octree(0)
    finally:
        A._LIB, A.LIB_PATH = keep


@pytest.fixture(scope="module")
def shim_and_ctx(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(d / "shim.c"), "-o", str(d / "shim.so"), "-ldl"], check=True)
    path = str(d / "liboctree_behind_shim.so")
    shutil.copy(A.LIB_PATH, path)
    shim = Shim(str(d / "shim.so"))
    ctx = context(path)
    assert shim.calls() > 0, "the copy does not allocate through the stand-in"
    yield shim, ctx
    shim.allow(-1)
    ctx.close()


def cloud():
    return np.random.default_rng(41).uniform(0.0, 10.0, (5000, 3))


def count(ctx, centers, radius, group=64):
    """Sphere counts in FP32 without the search counters."""
    counts = np.empty(len(centers), np.uint32)
    ctx.set_group(group)
    try:
        rc = ctx.L.oct_radius(ctx.h, A.K_SPHERE, A.A_STRUCT, A.PREC_FP32, centers.ctypes.data, None, None, radius, len(centers),
                              0, counts.ctypes.data, None)
    finally:
        ctx.set_group(-1)
    return rc, counts


def test_failed_rebuild_leaves_no_tree(shim_and_ctx):
    shim, ctx = shim_and_ctx
    xyz = cloud()
    sx, keys, _, c, r = O.sort_points(A.ENC_MORTON, xyz)
    centers = np.ascontiguousarray(sx[::50])
    _, want = O.radius(O.Tree(keys, 64, A.ENC_MORTON, c, r), sx, A.K_SPHERE, A.A_STRUCT, centers, 0.8)
    leaf, failures = 64, 0
    for allowed in range(12):
        ctx.set_points(xyz)
        ctx.sort_points(A.ENC_MORTON, fetch=False)
        ctx.build(leaf)
        rc, counts = count(ctx, centers, 0.8)
        assert rc == 0
        np.testing.assert_array_equal(counts, want)
        print(f"[gpu] rebuild with {allowed} allocations", flush=True)
        leaf = max(1, leaf // 2)  # smaller leaves: the node arrays grow
        shim.allow(allowed)
        try:
            ctx.build(leaf)
            rc, counts = count(ctx, centers, 0.8)
            assert rc == 0  # the rebuild had enough
            np.testing.assert_array_equal(counts, want)
        except A.OctError:
            failures += 1
            rc, _ = count(ctx, centers, 0.8)
            assert rc != 0 and b"before oct_build" in ctx.L.oct_last_error(ctx.h)
            with pytest.raises(A.OctError, match="before oct_build"):
                ctx.knn(3, idx=np.arange(4))
            with pytest.raises(A.OctError, match="before oct_build"):
                ctx.get_tree()
        finally:
            shim.allow(-1)
    assert failures > 0
    ctx.build(32)
    rc, counts = count(ctx, centers, 0.8)
    assert rc == 0
    np.testing.assert_array_equal(counts, want)


def test_counts_without_room_for_the_boxes(shim_and_ctx):
    """The tight boxes of a tree are allocated by its first count that can use them. Without room the cells are judged,
    and the counts that follow do not ask again until the next build."""
    shim, ctx = shim_and_ctx
    xyz = np.random.default_rng(42).uniform(0.0, 10.0, (60_000, 3))  # more nodes than the other test's trees
    sx, keys, _, c, r = O.sort_points(A.ENC_MORTON, xyz)
    centers = np.ascontiguousarray(sx[::500])
    _, want = O.radius(O.Tree(keys, 4, A.ENC_MORTON, c, r), sx, A.K_SPHERE, A.A_STRUCT, centers, 0.4)
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_MORTON, fetch=False)
    ctx.build(4)
    count(ctx, centers, 0.4, group=0)  # the buffers of the queries and results
    asked = []
    for allowed in (0, 0, 0):
        before = shim.calls()
        shim.allow(allowed)
        try:
            rc, counts = count(ctx, centers, 0.4)
        finally:
            shim.allow(-1)
        asked.append(shim.calls() - before)
        assert rc == 0, ctx.L.oct_last_error(ctx.h)
        np.testing.assert_array_equal(counts, want)
    print(f"[gpu] allocations of three counts: {asked}", flush=True)
    assert asked[0] > 0 and asked[1:] == [0, 0]
    before = shim.calls()
    ctx.build(4)
    rc, counts = count(ctx, centers, 0.4)
    assert rc == 0 and shim.calls() > before
    np.testing.assert_array_equal(counts, want)


def test_memory_the_boxes_keep(shim_and_ctx):
    """Of what the boxes are made from, only the boxes themselves stay allocated."""
    shim, ctx = shim_and_ctx
    xyz = np.random.default_rng(43).uniform(0.0, 20.0, (400_000, 3))
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_MORTON, fetch=False)
    ctx.build(16)
    centers = np.ascontiguousarray(xyz[:100])
    rc, want = count(ctx, centers, 0.5, group=0)
    assert rc == 0
    before = shim.calls()
    rc, counts = count(ctx, centers, 0.5)
    print(f"[gpu] allocations of the first count: {shim.calls() - before}", flush=True)
    assert rc == 0 and shim.calls() - before == 1
    np.testing.assert_array_equal(counts, want)
    perm, keys = ctx.sort_points(A.ENC_MORTON)[2:]  # the sort's buffers are its own again
    c, r = O.mbb(xyz)
    okeys, operm = O.sort(O.encode(A.ENC_MORTON, xyz, c, r))
    np.testing.assert_array_equal(keys, okeys)
    np.testing.assert_array_equal(perm, operm)


def test_pinned_pages_are_given_back(shim_and_ctx, tmp_path):
    """The contexts share a slab of pinned pages, 64 of them; those beyond have their own. All of it goes with the last
    context, and contexts made after that work."""
    shim, _ = shim_and_ctx
    path = str(tmp_path / "liboctree_pages.so")  # a copy of its own: no context of it lives yet
    shutil.copy(A.LIB_PATH, path)
    before = shim.pinned()
    xyz = cloud()
    for n in (1, 3, 66, 1):
        print(f"[gpu] {n} contexts", flush=True)
        ctxs = [context(path) for _ in range(n)]
        assert shim.pinned() - before == 1 + max(0, n - 64)
        for c in (ctxs[0], ctxs[-1]):
            c.set_points(xyz)
            c.sort_points(A.ENC_MORTON, fetch=False)
            c.build(64)
            rc, counts = count(c, np.ascontiguousarray(xyz[:10]), 0.5)
            assert rc == 0 and counts.min() > 0
        for c in ctxs[: n // 2]:
            c.close()
        assert shim.pinned() > before
        for c in ctxs[n // 2 :]:
            c.close()
        assert shim.pinned() == before
