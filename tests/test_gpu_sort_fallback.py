"""A partition sort that falls back to the LSD passes, whichever digit histograms the encode kernel left: it writes
those of the LSD passes only where the sort form chosen at that time takes them, and the form may be chosen anew
between the encode and the sort. Permutation and sorted keys are the oracle's (the stable sort by key)."""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu


def narrow_cluster(n, cluster, width, seed):
    """`cluster` points within `width` of each other among n spread over 1000: more than one workgroup sorts."""
    rng = np.random.default_rng(seed)
    xyz = 1000.0 * rng.random((n, 3))
    xyz[rng.permutation(n)[:cluster]] = 400.0 + width * rng.random((cluster, 3))
    return xyz


@pytest.mark.parametrize("encoded,sorted_as", [(0, 1), (0, 2), (1, 1), (1, 0), (2, 0), (0, 0), (None, 1), (0, None)])
@pytest.mark.parametrize("n,cluster,width", [(60_000, 40_000, 2.0), (300_000, 60_000, 0.001)])
@pytest.mark.parametrize("enc", [A.ENC_MORTON, A.ENC_HILBERT])
def test_form_chosen_between_encode_and_sort(ctx, enc, n, cluster, width, encoded, sorted_as):
    xyz = narrow_cluster(n, cluster, width, 7)
    c, r = O.mbb(xyz)
    keys, perm = O.sort(O.encode(enc, xyz, c, r))
    print(f"[sort fallback] n={n} enc={enc} encoded as {encoded}, sorted as {sorted_as}", flush=True)
    ctx.current = None
    try:
        for _ in range(2):  # the second time with what the first has learned of the points
            ctx.set_sort(encoded)
            ctx.set_points(xyz)
            ctx.encode(enc, c, r, fetch=False)
            ctx.set_sort(sorted_as)
            gperm, gkeys = ctx.sort()
            np.testing.assert_array_equal(gkeys, keys)
            np.testing.assert_array_equal(gperm, perm)
        ctx.encode(enc, c, r, fetch=False)  # the same points again
        gperm, gkeys = ctx.sort()
        np.testing.assert_array_equal(gkeys, keys)
        np.testing.assert_array_equal(gperm, perm)
    finally:
        ctx.set_sort(None)
