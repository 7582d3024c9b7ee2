"""GPU sort parity where the partition sort splits long 16-bit segments device-wide.

From 2^18 keys on, a 16-bit segment above max(4096, n / 1024) keys (at most 32768) is split by the next 8 bits
in one more device-wide pass; its pieces are sorted by one workgroup each, or split there again. Clouds:
one dense cluster among spread points, sized around the limit, above the 32768 keys a workgroup
takes, ordered along a line (runs of equal digits, as a moving scanner leaves them), several clusters that
share tiles of the pass, and a cluster too narrow for 24 bits to separate, which the LSD passes sort. Bar:
permutation and sorted keys bit-exact (the stable sort by key, reference point_encoder.hpp:285-383).
"""
import numpy as np
import pytest

import octree_amd as A
import pyoracle as O

pytestmark = pytest.mark.gpu

LIMIT = 1 << 18  # fewest keys with which the split runs


def cloud(clusters, n, width, seed, ordered=False):
    """`clusters` sizes, each inside a cube of side `width` at its own spot, with uniform points up to n."""
    rng = np.random.default_rng(seed)
    parts = []
    for c in clusters:
        t = np.sort(rng.random((c, 1)), axis=0) if ordered else rng.random((c, 3))
        parts.append(1000.0 * rng.random(3) + width * (t * np.ones(3)))
    parts.append(1000.0 * rng.random((n - sum(clusters), 3)))
    xyz = np.concatenate(parts)
    return xyz if ordered else xyz[rng.permutation(n)]


CASES = {
    "below_split_size": lambda: cloud([30_000], LIMIT - 1, 5.0, 1),
    "at_split_size": lambda: cloud([30_000], LIMIT, 5.0, 2),
    "piece_4096_4097": lambda: cloud([4096, 4097, 4098], LIMIT + 77, 2.0, 3),
    "one_tile_6144_6145": lambda: cloud([6144, 6145, 12288, 12289], LIMIT + 5, 2.0, 4),
    "cluster_200k": lambda: cloud([200_000], 300_001, 8.0, 5),
    "line_250k": lambda: cloud([250_000], 300_000, 10.0, 6, ordered=True),
    "many_clusters": lambda: cloud([9000 + 137 * i for i in range(24)], 600_000, 6.0, 7),
    "everything_one_segment": lambda: cloud([400_000 - 8], 400_000, 3.0, 8),
    "too_narrow_60k": lambda: cloud([60_000], 300_000, 0.001, 9),
    "duplicates": lambda: np.repeat(cloud([3000], 40_000, 4.0, 10), 8, axis=0),
}


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("enc", [A.ENC_MORTON, A.ENC_HILBERT])
@pytest.mark.parametrize("name", list(CASES))
def test_split_sort_matches_oracle(ctx, name, enc, mode):
    xyz = CASES[name]()
    print(f"[sort split] {name} n={len(xyz)} enc={enc} mode={mode}", flush=True)
    _, keys, perm, c, r = O.sort_points(enc, xyz)
    try:
        ctx.set_sort(mode)
        ctx.set_points(xyz)
        ctx.current = None
        gc, gr, gperm, gkeys = ctx.sort_points(enc)
    finally:
        ctx.set_sort(None)
    np.testing.assert_array_equal(gkeys, keys)
    np.testing.assert_array_equal(gperm, perm)
    np.testing.assert_array_equal(gc, c)


def test_repeated_splits(ctx):
    """From 2^26 keys on the split is repeated on the next two digits: a cluster whose 24-bit pieces are too long, and
    one that only 40 bits separate. The permutation is checked by what defines it."""
    n, big, narrow = (1 << 26) + 5, 20_000_000, 100_000
    rng = np.random.default_rng(12)
    xyz = 1000.0 * rng.random((n, 3))
    xyz[1000 : 1000 + big] = 321.0 + 5.0 * rng.random((big, 3))
    xyz[-narrow:] = 654.3 + 0.5 * rng.random((narrow, 3))
    print(f"[sort split] repeated n={n}", flush=True)
    ctx.set_points(xyz)
    ctx.current = None
    del xyz
    c, r = ctx.bbox()
    keys = ctx.encode(A.ENC_MORTON, c, r)
    perm, skeys = ctx.sort()
    seen = np.zeros(n, np.uint8)
    seen[perm] = 1
    assert seen.all()
    np.testing.assert_array_equal(skeys, keys[perm])
    up, same = skeys[1:] > skeys[:-1], skeys[1:] == skeys[:-1]
    assert (up | same).all()
    assert (perm[1:][same] > perm[:-1][same]).all()
    ctx.set_points(np.zeros((1, 3)))  # gives the memory's owner a small cloud for the tests that follow
    ctx.current = None
