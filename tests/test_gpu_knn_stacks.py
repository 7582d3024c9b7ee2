"""kNN among stacks of coincident points (returns without a range, all at the scanner, are such): thousands of points
at one distance from a query, far more than a query keeps. Neighbours are the brute-force ones, ties by index, also
where a stack met later holds smaller indices at the same distance; and the work stays that of the points tested."""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu

KS = (1, 7, 16, 31, 32, 64, 100, 128, 250, 500, 1024)


def built(ctx, xyz, enc, leaf):
    ctx.current = None
    ctx.set_points(xyz)
    _, _, perm, _ = ctx.sort_points(enc)
    ctx.build(leaf)
    return np.ascontiguousarray(xyz[perm.astype(np.int64)])


@pytest.mark.parametrize("enc", [A.ENC_MORTON, A.ENC_HILBERT])
@pytest.mark.parametrize("leaf", [16, 128])
def test_ties_by_index(ctx, leaf, enc):
    """Stacks of 1500 at the corners of a cube among other points; queries at the corners, at the cube's centre
    (eight stacks at one distance), on its faces and edges (four, two), and near them by less than FP32 resolves."""
    rng = np.random.default_rng(51)
    corners = np.stack(np.meshgrid(*[[10.0, 12.0]] * 3, indexing="ij"), -1).reshape(-1, 3)
    xyz = np.concatenate([np.repeat(corners, 1500, axis=0), rng.uniform(0.0, 24.0, (8000, 3))])
    xyz = xyz[rng.permutation(len(xyz))]
    sx = built(ctx, xyz, enc, leaf)
    q = np.concatenate([corners, [[11.0, 11.0, 11.0], [11.0, 11.0, 10.0], [11.0, 10.0, 10.0], [12.0, 12.0, 11.0]],
                        corners + rng.choice([-1.0, 1.0], (8, 3)) * 1e-9, rng.uniform(9.0, 13.0, (12, 3)), sx[:9]])
    for k in KS:
        bi, bd = O.knn_brute(sx, q, k)
        print(f"[stacks] k={k} leaf={leaf} enc={enc}", flush=True)
        for prec in (A.PREC_FP64, A.PREC_FP32):
            gi, gd, _ = ctx.knn(k, precision=prec, centers=q)
            np.testing.assert_array_equal(gi.astype(np.int64), bi, err_msg=f"k={k} prec={prec}")
            assert np.array_equal(gd.view(np.uint64), bd.view(np.uint64))


@pytest.mark.parametrize("k", [1, 10, 32, 100, 250])
def test_a_stack_costs_no_selection_per_step(ctx, k):
    """64 queries at a stack of 40 000: once the k-th is known exactly no further point of the stack is kept. A group
    of lanes then needs a few selections, where one every one to four steps of its 625 or more was made before."""
    rng = np.random.default_rng(52)
    xyz = np.concatenate([rng.uniform(0.0, 50.0, (20_000, 3)), np.repeat([[25.0, 25.0, 25.0]], 40_000, axis=0)])
    sx = built(ctx, xyz, A.ENC_MORTON, 64)
    q = np.full((64, 3), 25.0)
    bi, bd = O.knn_brute(sx, q[:1], k)
    print(f"[stacks] k={k}", flush=True)
    gi, gd, st = ctx.knn(k, centers=q)
    np.testing.assert_array_equal(gi.astype(np.int64), np.repeat(bi, 64, axis=0))
    np.testing.assert_array_equal(gd, np.repeat(bd, 64, axis=0))
    print(f"[stacks] k={k} selections of all waves {st['class_slots']}, steps {st['test_slots']}", flush=True)
    assert st["test_slots"] >= 40_000 // 64  # every point of the stack was tested
    assert st["class_slots"] <= 64 * 8  # eight per query
