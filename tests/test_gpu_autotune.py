"""The autotuner of the radius counts on samples far smaller than the cloud: what it stores is never far from the
fastest of the times it measured, however few queries the caller asked it to time."""
import pytest

import octree_amd as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tile():
    ctx = A.Octree(0)
    ctx.set_points(A.lidar_tile(3_000_000, seed=12, extent=250.0))
    ctx.sort_points(A.ENC_HILBERT)
    ctx.build(128)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("sample", [1, 500, 10_000, 1 << 17])
@pytest.mark.parametrize("kernel,algo,prec", [(A.K_SPHERE, A.A_STRUCT, A.PREC_FP32), (A.K_SPHERE, A.A_PRUNE, A.PREC_FP64),
                                              (A.K_CUBE, A.A_NEIGHBORS, A.PREC_FP64)])
def test_small_samples(tile, sample, kernel, algo, prec):
    print(f"[gpu] autotune kernel={kernel} algo={algo} prec={prec} sample={sample}", flush=True)
    best, ms = tile.autotune_radius(kernel, algo, prec, 1.5, sample_nq=sample)
    times = dict(zip((0, 16, 32, 64), [float(m) for m in (ms.values() if isinstance(ms, dict) else ms)]))
    print(best, times, flush=True)
    # a launch of at least two rounds of resident waves: its idle end is a fifth of it at most
    assert times[best] <= 1.25 * min(times.values())
    assert tile.tuned_radius(kernel, algo, prec) == best
