"""Result lists and group-kernel counts against the oracle where the kernels change shape: query counts around
a wave's 8 and 64 queries, leaves around the 16-point steps and 64-point chunks of the point tests, empty and
single-leaf trees, radii from nothing to the whole cloud. Every comparison is exact (lists entry for entry, in
the reference's emission order)."""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu

KERNELS = [A.K_SPHERE, A.K_CIRCLE, A.K_CUBE, A.K_SQUARE]
ALGOS = [A.A_NEIGHBORS, A.A_PRUNE, A.A_STRUCT]


@pytest.fixture(scope="module")
def ctx():
    c = A.Octree(0)
    yield c
    c.close()


def clouds():
    rng = np.random.default_rng(11)
    flat = rng.uniform(0, 10, (3000, 3)) * [1.0, 1.0, 0.02]
    clump = np.concatenate([rng.normal(0, 0.01, (400, 3)) + [3, 3, 3], rng.uniform(0, 8, (600, 3))])
    return {
        "one": np.array([[1.0, 2.0, 3.0]]),
        "root_leaf_17": rng.uniform(0, 1, (17, 3)),
        "root_leaf_130": rng.uniform(0, 1, (130, 3)),
        "flat": flat,
        "clump": clump,  # leaves of every size, many empty children, deep levels
    }


@pytest.mark.parametrize("name,leaf", [("one", 4), ("root_leaf_17", 17), ("root_leaf_130", 130), ("flat", 1), ("flat", 15),
                                       ("flat", 33), ("flat", 129), ("clump", 3), ("clump", 16), ("clump", 65)])
def test_lists_equal_the_oracle(ctx, name, leaf):
    xyz = clouds()[name]
    ctx.set_points(xyz)
    c, r, perm, keys = ctx.sort_points(A.ENC_HILBERT)
    ctx.build(leaf)
    sx, okeys, operm, oc, orad = O.sort_points(O.ENC_HILBERT, xyz)
    tree = O.Tree(okeys, leaf, O.ENC_HILBERT, oc, orad)
    n = len(sx)
    rng = np.random.default_rng(5)
    for nq in (1, 9, 65, 200):
        nq = min(nq, n)
        idx = np.sort(rng.choice(n, nq, replace=False)).astype(np.uint32)
        for radius in (0.0, 0.6, 50.0):
            for kernel in KERNELS:
                for algo in ALGOS:
                    ref, sizes = O.radius(tree, sx, kernel, algo, sx[idx.astype(np.int64)], radius)
                    for prec in (A.PREC_FP64, A.PREC_FP32):
                        tag = (name, leaf, nq, radius, kernel, algo, prec)
                        counts, lists, _ = ctx.radius(kernel, algo, prec, idx=idx, radius=radius, lists=True)
                        assert np.array_equal(counts, sizes), tag
                        assert all(np.array_equal(x, y) for x, y in zip(lists, ref)), tag
                        ctx.set_group(0)  # counts by the same traversal
                        counts, _ = ctx.radius(kernel, algo, prec, idx=idx, radius=radius)
                        ctx.set_group(-1)
                        assert np.array_equal(counts, sizes), tag


def dense_clouds():
    rng = np.random.default_rng(3)
    flat = rng.uniform(0, 60, (140_003, 3)) * [1.0, 1.0, 0.02]
    clump = np.concatenate([rng.normal(0, 0.02, (9_000, 3)) + [3, 3, 3], rng.uniform(0, 12, (131_001, 3))])
    return {"flat": flat, "clump": clump}


@pytest.mark.parametrize("name,leaf,radius", [("flat", 16, 0.4), ("flat", 130, 0.9), ("clump", 5, 0.3), ("clump", 64, 0.7)])
def test_shared_traversal_lists(ctx, name, leaf, radius):
    """More than 2^17 queries take the lists of 64 queries per wave (leaves tested in 64- or 48-point chunks, on
    the queries' own lanes or moved onto lane groups): equal to the same queries in calls small enough for the
    group kernel, and to the oracle on a sample."""
    xyz = dense_clouds()[name]
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_MORTON)
    ctx.build(leaf)
    sx, okeys, operm, oc, orad = O.sort_points(O.ENC_MORTON, xyz)
    tree = O.Tree(okeys, leaf, O.ENC_MORTON, oc, orad)
    n = len(sx)
    idx = np.arange(n, dtype=np.uint32)
    some = np.arange(7, n, 211)
    for kernel in KERNELS:
        for algo in ALGOS:
            ref, sizes = O.radius(tree, sx, kernel, algo, sx[some], radius)
            for prec in (A.PREC_FP64, A.PREC_FP32):
                tag = (name, leaf, radius, kernel, algo, prec)
                w = 2 if algo == A.A_STRUCT else 1
                counts, offs, ent, st = ctx.radius_csr(kernel, algo, prec, idx, radius)
                parts = [ctx.radius_csr(kernel, algo, prec, h, radius) for h in np.array_split(idx, 2)]
                assert np.array_equal(counts, np.concatenate([p[0] for p in parts])), tag
                assert np.array_equal(np.diff(offs), np.concatenate([np.diff(p[1]) for p in parts])), tag
                assert np.array_equal(ent, np.concatenate([p[2] for p in parts])), tag
                assert st["points_tested"] == sum(p[3]["points_tested"] for p in parts), tag
                assert st["nodes_classified"] == sum(p[3]["nodes_classified"] for p in parts), tag
                assert np.array_equal(counts[some], sizes), tag
                for q, r in zip(some, ref):
                    assert np.array_equal(ent[w * int(offs[q]):w * int(offs[q + 1])], np.asarray(r).reshape(-1)), tag


@pytest.mark.parametrize("stride", [17, 18])
def test_many_sparse_queries(ctx, stride):
    """More than 2^20 queries at one point in 17 or 18 share traversals (counts and lists); the same queries in calls
    of at most 2^17 go their own way. Equal counts and list sizes."""
    nq = (1 << 20) + 3
    rng = np.random.default_rng(stride)
    ctx.set_points(rng.uniform(0, 100, (nq * stride, 3)) * [1.0, 1.0, 0.05])
    ctx.sort_points(A.ENC_MORTON, fetch=False)
    ctx.build(64)
    idx = (np.arange(nq, dtype=np.uint64) * stride).astype(np.uint32)
    for algo in (A.A_PRUNE, A.A_STRUCT):
        print(f"[lists] {nq} queries, one point in {stride}, algo={algo}", flush=True)
        counts, _ = ctx.radius(A.K_SPHERE, algo, A.PREC_FP32, idx=idx, radius=0.3)
        listed = np.empty(nq, np.uint32)
        rc = ctx.L.oct_radius(ctx.h, A.K_SPHERE, algo, A.PREC_FP32, None, idx.ctypes.data, None, 0.3, nq, 1, listed.ctypes.data, None)
        assert rc == 0
        np.testing.assert_array_equal(listed, counts)
        for a in range(0, nq, 1 << 19):  # a part of each half million, one small call
            part = idx[a : a + 4001]
            few, _ = ctx.radius(A.K_SPHERE, algo, A.PREC_FP32, idx=part, radius=0.3)
            np.testing.assert_array_equal(counts[a : a + 4001], few)
