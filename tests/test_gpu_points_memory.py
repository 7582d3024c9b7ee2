"""Points given to the device entry point from memory that is not the context's device's own: the runtime's copy takes
them or refuses them, as before the copy kernel; no kernel reads them."""
import ctypes as C

import numpy as np
import pytest

import octree_amd as A
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def given(ctx, ptr, n):
    ctx.current = None
    ctx.n = n
    rc = ctx.L.oct_set_points_dev(ctx.h, ptr, n, 24)
    return rc, ctx.sort_points(A.ENC_HILBERT) if rc == 0 else None


@pytest.mark.parametrize("n", [1, 1000, 300_001])
def test_pinned_and_pageable_host_memory(ctx, n):
    xyz = np.random.default_rng(n).normal(0.0, 30.0, (n, 3))
    ctx.current = None
    ctx.set_points(xyz)
    want = ctx.sort_points(A.ENC_HILBERT)
    hip = Hip().h
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    pinned = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(pinned), xyz.nbytes, 0) == 0
    try:
        C.memmove(pinned, xyz.ctypes.data, xyz.nbytes)
        print(f"[gpu] pinned points n={n}", flush=True)
        rc, got = given(ctx, pinned, n)
        assert rc == 0
        for x, y in zip(got, want):
            np.testing.assert_array_equal(x, y)
    finally:
        hip.hipHostFree(pinned)
    plain = np.empty(3 * n + 2)
    plain = plain[(-plain.ctypes.data // 8) % 2 :][: 3 * n]  # 16-byte aligned
    plain[:] = xyz.reshape(-1)
    print(f"[gpu] pageable points n={n}", flush=True)
    rc, got = given(ctx, plain.ctypes.data, n)
    if rc == 0:
        for x, y in zip(got, want):
            np.testing.assert_array_equal(x, y)
    ctx.set_points(xyz)  # whichever way it ended, the context goes on
    for x, y in zip(ctx.sort_points(A.ENC_HILBERT), want):
        np.testing.assert_array_equal(x, y)
