"""The two forms of a batch's device radius pass: sparse queries by their own traversal (8 lanes each), more than
2^17 queries that cover the clouds by one traversal per 64. Both sides of the line, every kernel and both
precisions; clouds of very different sizes (an empty one, a single point, a root leaf), a query count per cloud
that leaves ragged tiles. Counts equal oct_batch_radius's, which the oracle checks elsewhere."""
import numpy as np
import pytest

import octree_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr", [1, 63, 20_001, (1 << 17) + 1])
def test_radius_pass_forms(nr):
    rng = np.random.default_rng(nr)
    sizes = [0, 1, 20, 300, 5_000, 150_003]
    clouds = [rng.uniform(0, 20, (n, 3)) * [1.0, 1.0, 0.1] + 100.0 * i for i, n in enumerate(sizes)]
    live = np.array([i for i, n in enumerate(sizes) if n])
    rc = rng.choice(live, nr, p=[0.01, 0.04, 0.1, 0.25, 0.6]).astype(np.uint32)
    ri = (rng.random(nr) * np.array(sizes)[rc]).astype(np.uint32)
    rr = rng.choice([0.0, 0.05, 0.3, 30.0], nr, p=[0.1, 0.5, 0.399, 0.001])
    kc, ki, kk = live[-1:].astype(np.uint32), np.array([7], np.uint32), np.array([5], np.uint32)
    b = A.Batch(0)
    try:
        for i, xyz in enumerate(clouds):
            b.add(xyz, A.ENC_HILBERT if i % 2 else A.ENC_MORTON, 32)
        b.queries(rc, ri, rr, kc, ki, kk, kmax=8)
        for kernel in (A.K_SPHERE, A.K_CIRCLE, A.K_CUBE, A.K_SQUARE):
            for prec in (A.PREC_FP64, A.PREC_FP32):
                algo = (A.A_STRUCT, A.A_PRUNE, A.A_NEIGHBORS)[kernel % 3]
                print(f"[batch forms] nr={nr} kernel={kernel} algo={algo} prec={prec}", flush=True)
                b.pipeline(kernel, algo, prec, graph=True)
                b.pipeline(kernel, algo, prec, graph=True)  # a replay
                counts = b.pipeline_results()[0]
                ref, _ = b.radius(kernel, algo, prec, rc, ri, rr)
                np.testing.assert_array_equal(counts, ref)
    finally:
        b.close()
