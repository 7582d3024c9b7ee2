"""Counts asked for without the search counters (the only calls that judge children by the tight boxes of their
points and test leaves on the matrix cores with that judgement behind them) and lists, where the forms could
disagree: points outside the cells their keys name. Every form returns exactly the oracle's results."""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu

GROUPS = (0, 16, 32, 64)


@pytest.fixture(scope="module")
def ctx():
    c = A.Octree(0)
    yield c
    c.close()


def count(ctx, kernel, algo, prec, centers, radii):
    """Counts without the search counters."""
    centers = np.ascontiguousarray(centers)
    radii = np.ascontiguousarray(radii)
    counts = np.empty(len(centers), np.uint32)
    rc = ctx.L.oct_radius(ctx.h, kernel, algo, prec, centers.ctypes.data, None, radii.ctypes.data, 0.0, len(centers), 0,
                          counts.ctypes.data, None)
    assert rc == 0, ctx.L.oct_last_error(ctx.h)
    return counts


def check_forms(ctx, sx, tree, centers, radii, kernels, tag, algos=(A.A_NEIGHBORS, A.A_PRUNE, A.A_STRUCT), lists=True):
    for kernel in kernels:
        for algo in algos:
            ref, sizes = O.radius(tree, sx, kernel, algo, centers, radii)
            for prec in (A.PREC_FP64, A.PREC_FP32):
                if lists:
                    counts, got, _ = ctx.radius(kernel, algo, prec, centers=centers, radii=radii, lists=True)
                    np.testing.assert_array_equal(counts, sizes, err_msg=f"{tag} list sizes k={kernel} a={algo} p={prec}")
                    for q in range(len(centers)):
                        assert np.array_equal(got[q], ref[q]), f"{tag} list k={kernel} a={algo} p={prec} query {q}"
                for g in GROUPS:
                    print(f"[forms] {tag} kernel={kernel} algo={algo} prec={prec} G={g}", flush=True)
                    ctx.set_group(g)
                    try:
                        counts = count(ctx, kernel, algo, prec, centers, radii)
                        np.testing.assert_array_equal(counts, sizes, err_msg=f"{tag} k={kernel} a={algo} p={prec} G={g}")
                        counts, _ = ctx.radius(kernel, algo, prec, centers=centers, radii=radii)
                        np.testing.assert_array_equal(counts, sizes, err_msg=f"{tag} with counters k={kernel} a={algo} p={prec} G={g}")
                    finally:
                        ctx.set_group(-1)


def cloud(seed=31):
    """A cloud with queries in it and around it, their radii from a leaf's size to the cloud's."""
    rng = np.random.default_rng(seed)
    xyz = np.concatenate([rng.uniform(0.0, 20.0, (2500, 3)), rng.normal(10.0, 0.4, (700, 3))])
    centers = np.concatenate([xyz[rng.permutation(len(xyz))[:150]], rng.uniform(-6.0, 26.0, (50, 3))])
    return xyz, centers, rng.choice([0.4, 1.5, 4.0, 9.0], len(centers))


@pytest.mark.parametrize("shrink", [0.999, 0.7, 0.3])
@pytest.mark.parametrize("enc", [A.ENC_MORTON, A.ENC_HILBERT])
def test_encoded_with_a_box_smaller_than_the_cloud(ctx, enc, shrink):
    """Points outside the box are clamped into its outermost cells, far from where they are: an OUTSIDE cell drops
    them and an INSIDE one counts them, whatever their distance."""
    xyz, centers, radii = cloud()
    c, r = O.mbb(xyz)
    r = r * shrink
    keys = O.encode(enc, xyz, c, r)
    sk, perm = O.sort(keys)
    sx = np.ascontiguousarray(xyz[perm.astype(np.int64)])
    ctx.set_points(xyz)
    ctx.encode(enc, c, r)
    gperm, gkeys = ctx.sort()
    np.testing.assert_array_equal(gkeys, sk)
    ctx.build(24)
    check_forms(ctx, sx, O.Tree(sk, 24, enc, c, r), centers, radii, (A.K_SPHERE, A.K_CUBE), f"shrink={shrink} enc={enc}")


@pytest.mark.parametrize("enc", [A.ENC_MORTON, A.ENC_HILBERT])
def test_sorted_clouds_whose_codes_are_not_their_points(ctx, enc):
    """Codes of a moved copy of part of the cloud, or of a box that lies elsewhere."""
    xyz, centers, radii = cloud(32)
    c, r = O.mbb(xyz)
    rng = np.random.default_rng(5)
    moved = xyz.copy()
    some = rng.permutation(len(xyz))[:300]
    moved[some] += rng.normal(0.0, 0.7, (300, 3))
    for tag, src, cc in (("moved", moved, c), ("box elsewhere", xyz, c + [2.0, 0.0, -1.0])):
        sk, perm = O.sort(O.encode(enc, src, cc, r))
        sx = np.ascontiguousarray(xyz[perm.astype(np.int64)])
        ctx.set_sorted(sx, sk, enc, cc, r)
        ctx.build(24)
        check_forms(ctx, sx, O.Tree(sk, 24, enc, cc, r), centers, radii, (A.K_SPHERE, A.K_CUBE), f"{tag} enc={enc}")
