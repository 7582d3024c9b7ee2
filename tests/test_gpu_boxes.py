"""Sphere counts with 64 queries per wave (FP32, algorithms Prune and Struct): children judged by the tight boxes
of their points, leaves tested on the matrix cores, ties decided by the walk from the root. Counts are exactly
the oracle's, where this can go wrong: a decimal lattice (distances equal to the radius up to the last bit, at
node corners as well), coordinates far from the origin, flat and clumped clouds, duplicates (leaves of more
than one 64-point chunk at the deepest level), leaf sizes around the 16-point rows, query sets around the
16-query tiles, per-query radii with zero and negative ones, and queries outside the cloud."""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = A.Octree(0)
    yield c
    c.close()


def lattice(step, n, offset):
    g = np.arange(n) * step
    return np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + offset


def clouds():
    rng = np.random.default_rng(21)
    flat = rng.uniform(0, 40, (6000, 3)) * [1.0, 1.0, 0.01]
    return {
        "lattice": (lattice(0.1, 17, 0.0), [0.1, 0.5, 0.7, 1.6, 5.0]),
        "lattice_far": (lattice(0.1, 13, [512345.6, 4765432.1, 103.7]), [0.1, 0.3, 0.5, 1.2]),
        "flat": (flat, [0.02, 0.8, 3.0, 100.0]),
        "flat_far": (flat + [480000.0, 5200000.0, 250.0], [0.02, 0.8, 3.0]),
        "clump": (np.concatenate([rng.normal(0, 0.01, (700, 3)) + 3.0, rng.uniform(0, 8, (1500, 3))]), [0.005, 0.05, 1.0]),
        "duplicates": (np.repeat(rng.uniform(0, 5, (30, 3)), 70, axis=0), [0.5, 2.0]),
        "tiny_radius": (rng.uniform(0, 1, (2000, 3)) + [1e6, 2e6, 0.0], [1e-9, 1e-4, 0.2]),
    }


def count(ctx, algo, centers, radius=0.0, radii=None):
    """Counts without the search counters (with them the octree cells are judged)."""
    centers = np.ascontiguousarray(centers)
    counts = np.empty(len(centers), np.uint32)
    rad = None if radii is None else np.ascontiguousarray(radii).ctypes.data
    rc = ctx.L.oct_radius(ctx.h, A.K_SPHERE, algo, A.PREC_FP32, centers.ctypes.data, None, rad, float(radius), len(centers), 0,
                          counts.ctypes.data, None)
    assert rc == 0, ctx.L.oct_last_error(ctx.h)
    return counts


def built(ctx, xyz, enc, leaf):
    sx, keys, perm, c, r = O.sort_points(enc, xyz)
    ctx.set_points(xyz)
    ctx.sort_points(enc)
    ctx.build(leaf)
    return sx, O.Tree(keys, leaf, enc, c, r)


@pytest.mark.parametrize("leaf", [1, 16, 17, 130])
@pytest.mark.parametrize("name", sorted(clouds()))
def test_counts_equal_the_oracle(ctx, name, leaf):
    xyz, radii = clouds()[name]
    for enc in (A.ENC_MORTON, A.ENC_HILBERT):
        sx, tree = built(ctx, xyz, enc, leaf)
        rng = np.random.default_rng(leaf)
        c = sx.mean(axis=0)
        outside = c + (sx[rng.integers(0, len(sx), 40)] - c) * 3.0
        centers = np.concatenate([sx[rng.permutation(len(sx))[:317]], outside])
        ctx.set_group(64)
        try:
            for r in radii:
                for algo in (A.A_PRUNE, A.A_STRUCT):
                    _, sizes = O.radius(tree, sx, A.K_SPHERE, algo, centers, r)
                    for nq in (1, 15, 16, 17, 64, len(centers)):
                        print(f"[boxes] {name} leaf={leaf} enc={enc} r={r} algo={algo} nq={nq}", flush=True)
                        counts = count(ctx, algo, centers[:nq], r)
                        np.testing.assert_array_equal(counts, sizes[:nq])
        finally:
            ctx.set_group(-1)


@pytest.mark.parametrize("name", ["flat", "lattice"])
def test_per_query_radii(ctx, name):
    xyz, _ = clouds()[name]
    sx, tree = built(ctx, xyz, A.ENC_HILBERT, 16)
    rng = np.random.default_rng(8)
    centers = sx[rng.permutation(len(sx))[:500]]
    radii = rng.choice([0.0, 0.1, 0.5, 2.0, -0.5, -1e-12, 1e-8], len(centers))
    radii[:128] = rng.choice([0.1, 0.7, 3.0], 128)  # waves without the odd ones
    ctx.set_group(64)
    try:
        for algo in (A.A_PRUNE, A.A_STRUCT):
            print(f"[boxes] per-query radii {name} algo={algo}", flush=True)
            _, sizes = O.radius(tree, sx, A.K_SPHERE, algo, centers, radii)
            counts = count(ctx, algo, centers, radii=radii)
            np.testing.assert_array_equal(counts, sizes)
    finally:
        ctx.set_group(-1)
