"""Points given as a device buffer: the copy takes the bounding box's first reduction on its way (16-byte words,
so an odd count ends in half a word, and an 8-byte aligned buffer takes the plain copy). Box, keys and permutation
must be those of the same points given from the host, NaN and infinite coordinates and signed zeros included."""
import numpy as np
import pytest

import octree_amd as A

pytestmark = pytest.mark.gpu


def from_host(ctx, xyz):
    ctx.set_points(xyz)
    return ctx.sort_points(A.ENC_HILBERT)


@pytest.mark.parametrize("n", [1, 2, 3, 127, 128, 129, 511, 513, 4097, 393_217, 786_433])
def test_device_points_equal_host_points(ctx, n):
    rng = np.random.default_rng(n)
    xyz = rng.normal(0.0, 50.0, (n, 3)) + [1000.0, -20.0, 0.0]
    clouds = [xyz]
    if n > 100:
        odd = xyz.copy()
        odd[rng.integers(0, n, 5), rng.integers(0, 3, 5)] = np.nan
        odd[-1, 2] = 1e6  # the last coordinate is the largest
        odd[0, 0] = -1e6
        clouds.append(odd)
        clouds.append(np.where(rng.random((n, 3)) < 0.5, 0.0, -0.0))
    ctx.current = None
    for c, cloud in enumerate(clouds):
        want = from_host(ctx, cloud)
        for off in (0, 1):  # element offset: 16- and 8-byte aligned
            buf = A.DeviceArray(np.concatenate([np.zeros(off), cloud.reshape(-1)]))
            try:
                ctx.n = n
                assert ctx.L.oct_set_points_dev(ctx.h, buf.ptr(off), n, 24) == 0
                box = ctx.bbox()
                got = ctx.sort_points(A.ENC_HILBERT)
            finally:
                buf.close()
            for x, y in zip(got, want):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (n, c, off)
            assert np.array_equal(box[0], want[0], equal_nan=True) and np.array_equal(box[1], want[1], equal_nan=True)
