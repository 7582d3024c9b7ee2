"""Radius searches on both sides of the limits between a traversal of its own for every query and one shared by 64:
more than 2^17 queries at one point in 16, more than 2^20 at one in 48 (lists) and one in 64 (counts). Counts are
asked for without the search counters, as a program does; they equal those of both forms chosen by hand. A list is
the same whichever side of a limit its call falls on."""
import numpy as np
import pytest

import octree_amd as A

pytestmark = pytest.mark.gpu

N = 70_000_000
RADIUS = 0.55
FEW, MANY = (1 << 17) + 77, (1 << 20) + 33


@pytest.fixture(scope="module")
def box():
    ctx = A.Octree(0)
    ctx.set_points(A.uniform_box(N, seed=8, size=(300.0, 300.0, 60.0)))
    ctx.sort_points(A.ENC_HILBERT, fetch=False)
    ctx.build(64)
    yield ctx
    ctx.close()


def count(ctx, prec, idx):
    out = np.empty(len(idx), np.uint32)
    rc = ctx.L.oct_radius(ctx.h, A.K_SPHERE, A.A_STRUCT, prec, None, idx.ctypes.data, None, RADIUS, len(idx), 0,
                          out.ctypes.data, None)
    assert rc == 0, ctx.L.oct_last_error(ctx.h)
    return out


def lists(ctx, algo, idx):
    counts = np.empty(len(idx), np.uint32)
    rc = ctx.L.oct_radius(ctx.h, A.K_SPHERE, algo, A.PREC_FP32, None, idx.ctypes.data, None, RADIUS, len(idx), 1,
                          counts.ctypes.data, None)
    assert rc == 0, ctx.L.oct_last_error(ctx.h)
    offs = np.empty(len(idx) + 1, np.uint64)
    assert ctx.L.oct_radius_fetch(ctx.h, offs.ctypes.data, None, 0) == 0
    words = int(offs[-1]) * (2 if algo == A.A_STRUCT else 1)
    ent = np.empty(words, np.uint32)
    assert ctx.L.oct_radius_fetch(ctx.h, offs.ctypes.data, ent.ctypes.data, words) == 0
    return counts, offs, ent


def strided(nq, stride):
    """nq queries, one point in `stride` exactly: the last one is moved so that they span nq * stride points."""
    idx = np.arange(nq, dtype=np.int64) * stride
    idx[-1] += stride - 1
    return idx.astype(np.uint32)


@pytest.mark.parametrize("nq,stride", [(FEW - 77, 1), (FEW, 1), (FEW, 16), (FEW, 17), (MANY, 48), (MANY, 49), (MANY, 64), (MANY, 65)])
def test_counts(box, nq, stride):
    idx = strided(nq, stride)
    for prec in (A.PREC_FP32, A.PREC_FP64):
        print(f"[dispatch] counts nq={nq} stride={stride} prec={prec}", flush=True)
        got = count(box, prec, idx)
        for g in (0, 64):
            box.set_group(g)
            try:
                np.testing.assert_array_equal(got, count(box, prec, idx))
            finally:
                box.set_group(-1)
        assert got.min() >= 1 and got.mean() > 4


@pytest.mark.parametrize("algo", [A.A_PRUNE, A.A_STRUCT])
@pytest.mark.parametrize("nq,stride", [(FEW, 16), (MANY, 48)])
def test_lists(box, nq, stride, algo):
    shared = strided(nq, stride)
    own = np.append(shared, np.uint32(N - 1))  # the same and one far away: too sparse to share
    print(f"[dispatch] lists nq={nq} stride={stride} algo={algo}", flush=True)
    c1, o1, e1 = lists(box, algo, shared)
    c2, o2, e2 = lists(box, algo, own)
    np.testing.assert_array_equal(c1, c2[:-1])
    np.testing.assert_array_equal(o1, o2[:-1])
    np.testing.assert_array_equal(e1, e2[: len(e1)])
    np.testing.assert_array_equal(c1, count(box, A.PREC_FP64, shared))
