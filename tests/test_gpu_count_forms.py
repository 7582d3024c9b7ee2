"""Counts asked for without the search counters (the only calls that judge children by the tight boxes of their
points and test leaves on the matrix cores with that judgement behind them) and lists, where the forms could
disagree: points outside the cells their keys name, points beyond FP32 and below it, NaNs. Every form returns
exactly the oracle's results."""
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


# ---- magnitudes at which the FP32 terms of a leaf overflow, or are not numbers
def spread_cloud(extent, far, seed=33):
    """200 points of a cluster around the box's centre, 1e-7 of the extent wide, and `far` over the whole extent: the
    root's children are leaves whose points are mostly far from the leaf's centre."""
    rng = np.random.default_rng(seed)
    near = rng.normal(0.0, 1e-7 * extent, (200, 3))
    corners = extent * np.array([[1.0, 1.0, 1.0], [-1.0, -1.0, -1.0]])
    xyz = np.concatenate([near, rng.uniform(-extent, extent, (far, 3)), corners])
    return xyz, np.concatenate([np.zeros((1, 3)), near[:40], near[:80] * 0.3]), xyz[-20:]


@pytest.mark.parametrize("extent", [1e14, 4e14, 1e15, 1e18, 6e19, 1e20, 1e24, 1e30])
@pytest.mark.parametrize("far", [3, 198])
def test_leaves_beyond_fp32_around_the_box_centre(ctx, extent, far):
    xyz, middle, outer = spread_cloud(extent, far)
    for enc in (A.ENC_MORTON, A.ENC_HILBERT):
        sx, keys, _, c, r = O.sort_points(enc, xyz)
        ctx.set_points(xyz)
        ctx.sort_points(enc)
        ctx.build(128)
        tree = O.Tree(keys, 128, enc, c, r)
        for where, centers in (("middle", middle), ("outer", outer)):  # not in one wave
            for rel in (1e-7, 0.3):
                check_forms(ctx, sx, tree, centers, np.full(len(centers), rel * extent), (A.K_SPHERE, A.K_CIRCLE),
                            f"extent={extent:g} far={far} {where} r={rel:g} enc={enc}", lists=False)


@pytest.mark.parametrize("ml", [16, 200])
@pytest.mark.parametrize("sign", ["positive", "negative", "both"])
def test_points_that_are_not_numbers(ctx, sign, ml):
    """NaN coordinates of either sign take the largest key: one deep leaf of them, and ordinary points of the box's
    last corner in it where the leaves are large."""
    rng = np.random.default_rng(34)
    xyz = rng.uniform(0.0, 8.0, (3000, 3))
    bits = {"positive": [0x7FF8000000000000], "negative": [0xFFF8000000000000],
            "both": [0x7FF8000000000000, 0xFFF8000000000000]}[sign]
    nan = np.array(bits, np.uint64).view(np.float64)
    odd = np.concatenate([np.arange(40), rng.permutation(3000)[:60]])
    xyz[odd] = rng.choice(nan, (len(odd), 1)) * np.ones((1, 3))
    xyz[odd[::3], 0] = 7.9  # not numbers on two axes
    good = xyz[~np.isnan(xyz).any(axis=1)]
    centers = np.concatenate([good[rng.permutation(len(good))[:150]], rng.uniform(7.0, 8.5, (50, 3))])
    for enc in (A.ENC_MORTON, A.ENC_HILBERT):
        sx, keys, _, c, r = O.sort_points(enc, xyz)
        ctx.set_points(xyz)
        ctx.sort_points(enc)
        ctx.build(ml)
        check_forms(ctx, sx, O.Tree(keys, ml, enc, c, r), centers, rng.choice([0.3, 1.0, 3.0], len(centers)),
                    (A.K_SPHERE, A.K_CIRCLE), f"NaN {sign} leaf={ml} enc={enc}", lists=False)


# ---- magnitudes at which the FP32 terms of a leaf vanish
@pytest.mark.parametrize("scale", [1e-15, 1e-18, 1e-20, 1e-21, 1e-22, 3e-23, 1e-24])
def test_leaves_below_fp32(ctx, scale):
    rng = np.random.default_rng(35)
    xyz = rng.uniform(-1.0, 1.0, (1500, 3)) * scale
    centers = np.concatenate([xyz[:100], rng.uniform(-1.2, 1.2, (30, 3)) * scale])
    sx, keys, _, c, r = O.sort_points(A.ENC_HILBERT, xyz)
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_HILBERT)
    ctx.build(64)
    check_forms(ctx, sx, O.Tree(keys, 64, A.ENC_HILBERT, c, r), centers, rng.choice([0.1, 0.4, 0.8], len(centers)) * scale,
                (A.K_SPHERE, A.K_CIRCLE), f"scale={scale:g}")


def test_the_first_count_reports_the_boxes_it_makes(ctx):
    """A tree's first count that uses the tight boxes makes them, over every node; its stage time says so."""
    xyz = np.random.default_rng(36).uniform(0.0, 50.0, (1_000_000, 3))
    centers = np.full((64, 3), 500.0)  # outside the root: the search itself is next to nothing
    radii = np.full(64, 0.3)
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_MORTON, fetch=False)
    times = []
    ctx.set_group(64)
    try:
        for _ in range(3):  # trees; the first one's count also loads code and allocates
            ctx.build(8)
            tree = []
            for _ in range(4):
                count(ctx, A.K_SPHERE, A.A_STRUCT, A.PREC_FP32, centers, radii)
                tree.append(ctx.stage_times()["search"])
            times.append(tree)
    finally:
        ctx.set_group(-1)
    print(f"[forms] search stage, four counts of each of three trees: {times}", flush=True)
    for tree in times[1:]:
        assert tree[0] > 3.0 * max(tree[1:])


# ---- radii whose squares, or whose boxes, leave FP64
@pytest.mark.parametrize("radius", [1e150, 1e155, 1e200, 9e299, 1.1e300, 1.7e308, np.inf])
def test_radii_beyond_fp64(ctx, radius):
    """Every point is a neighbour, none twice, and nothing but points."""
    rng = np.random.default_rng(37)
    xyz = rng.uniform(0.0, 10.0, (700, 3))
    centers = np.concatenate([xyz[:70], [[-50.0, 3.0, 1e5]]])
    radii = np.full(len(centers), radius)
    radii[::7] = 2.0
    sx, keys, _, c, r = O.sort_points(A.ENC_MORTON, xyz)
    ctx.set_points(xyz)
    ctx.sort_points(A.ENC_MORTON)
    ctx.build(64)
    check_forms(ctx, sx, O.Tree(keys, 64, A.ENC_MORTON, c, r), centers, radii,
                (A.K_SPHERE, A.K_CIRCLE, A.K_CUBE, A.K_SQUARE), f"radius={radius:g}")
