"""Ordered compaction of the coordinate steps at the edges of its runs (whole
multiples of 1,024 items, at most 1,024 runs): one item, one run less and more
an item, runs longer than 1,024 items, nothing and everything flagged.  Rows
are whole numbers in the input's order, so they equal the reference exactly.
"""
import numpy as np
import pytest

from helpers import prune_brute_force

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 1, 1023), (1, 1024, 1), (5, 5, 41), (3, 683, 1),
                                   (1024, 1024, 1), (1, 1, 1048577), (97, 101, 223)])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_occupancy_runs(s3dx, shape, share):
    rng = np.random.default_rng(7)
    occ = np.where(rng.random(shape) < share, 1.0, -1.0).astype(np.float32)
    if share == 0.3:
        occ.flat[0] = np.inf
        occ.flat[-1] = np.nan  # NaN > 0 is false
    n, rows = s3dx.occupancy_coords(s3dx.DeviceArray.from_host(occ), shape)
    print(f"occupancy {shape} share={share} n={n}", flush=True)
    want = np.argwhere(occ > 0).astype(np.int32)
    want = np.concatenate([np.zeros((want.shape[0], 1), np.int32), want], 1)
    assert n == want.shape[0]
    assert np.array_equal(rows.download()[:n], want)


def _cloud(n, seed):
    # Voxels of a box about twice the set, in no order, some rows twice, some
    # coordinates negative, two batches.
    rng = np.random.default_rng(seed)
    side = max(1, int(round((2 * n) ** (1 / 3))))
    c = rng.integers(0, side, (n, 4)).astype(np.int32) - side // 3
    c[:, 0] = rng.integers(0, 2, n)
    return c


@pytest.mark.parametrize("n", [1, 2, 5, 255, 257, 1023, 1024, 1025, 33001, 1048576, 1050000])
def test_prune_and_downsample_runs(s3dx, O, n):
    c = _cloud(n, n)
    d = s3dx.DeviceArray.from_host(c)
    got, rows = s3dx.prune_surface(d, n)
    print(f"prune n={n} -> {got}", flush=True)
    want = O.prune_surface(c)
    if n <= 1025:
        assert np.array_equal(want, prune_brute_force(c))
    assert got == want.shape[0]
    assert np.array_equal(rows.download()[:got], want)
    for most in (max(1, n - 1), max(1, n // 11)):
        want = O.downsample_coords(c, most)
        got, rows = s3dx.downsample_coords(d, n, most)
        print(f"downsample n={n} most={most} -> {got}", flush=True)
        assert got == want.shape[0]
        assert np.array_equal(rows.download()[:got], want)
