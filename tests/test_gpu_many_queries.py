"""Calls of 2^29 queries and more, whose launches of 8 lanes per query exceed one HIP grid: kNN and the counts of the
group kernel over a small cloud, the queries being its points over and over, so every result is known."""
import numpy as np
import pytest

import octree_amd as A
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

POINTS = 1021  # a prime: no launch boundary falls on the cloud's first point
QUERIES = (1 << 29) + 11


@pytest.fixture(scope="module")
def setup():
    ctx = A.Octree(0)
    ctx.set_points(np.random.default_rng(3).uniform(0.0, 10.0, (POINTS, 3)))
    ctx.sort_points(A.ENC_MORTON)
    ctx.build(16)
    hip = Hip()
    idx = hip.put(np.resize(np.arange(POINTS, dtype=np.uint32), QUERIES))
    yield ctx, hip, idx
    hip.free()
    ctx.close()


def check_repeats(hip, buf, want):
    """The device buffer holds `want` over and over."""
    got = hip.get(buf, QUERIES, want.dtype)
    whole = QUERIES // POINTS * POINTS
    assert (got[:whole].reshape(-1, POINTS) == want).all()
    assert (got[whole:] == want[: QUERIES - whole]).all()


def test_knn(setup):
    ctx, hip, idx = setup
    out, d2 = hip.alloc(4 * QUERIES), hip.alloc(4 * QUERIES)
    print(f"[gpu] kNN of {QUERIES} queries", flush=True)
    rc = ctx.L.oct_knn_dev(ctx.h, A.PREC_FP64, idx, 0, QUERIES, 1, out, d2, None)
    assert rc == 0, ctx.L.oct_last_error(ctx.h)
    ctx.synchronize()
    check_repeats(hip, out, np.arange(POINTS, dtype=np.int32))  # every point is its own nearest
    check_repeats(hip, d2, np.zeros(POINTS, np.float32))


def test_group_counts(setup):
    ctx, hip, idx = setup
    want, _ = ctx.radius(A.K_SPHERE, A.A_PRUNE, A.PREC_FP64, radius=0.4)
    counts = hip.alloc(4 * QUERIES)
    ctx.set_group(0)
    try:
        print(f"[gpu] counts of {QUERIES} queries", flush=True)
        rc = ctx.L.oct_radius_dev(ctx.h, A.K_SPHERE, A.A_PRUNE, A.PREC_FP64, idx, 0.4, QUERIES, counts, None)
        assert rc == 0, ctx.L.oct_last_error(ctx.h)
        ctx.synchronize()
    finally:
        ctx.set_group(-1)
    check_repeats(hip, counts, want)
