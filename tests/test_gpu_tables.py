"""Subdivide's one grid over the parents and coarsen's window path at the edges
of their blocks (8 and 32 parents; 64 rows a wave, 1,024 a block).  Whole
numbers, equal to the oracle's; a map that is not 16-byte aligned takes the
general kernels.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _set(n, seed, ordered):
    rng = np.random.default_rng(seed)
    side = max(2, int(np.ceil((3 * n) ** (1 / 3))))
    cells = rng.choice(side ** 3, n, replace=False)
    cells = np.sort(cells) if ordered else cells
    c = np.stack([0 * cells, cells // side ** 2, cells // side % side, cells % side], 1)
    return np.ascontiguousarray(c.astype(np.int32))


@pytest.mark.parametrize("p", [1, 7, 8, 9, 31, 32, 33, 257, 8 * 32 * 8 + 5])
def test_subdivide_blocks(s3dx, O, p):
    c = _set(p, p, False)
    if p > 8:
        c[:, 1:] -= 3  # negative parents
    d = s3dx.DeviceArray.from_host(c)
    child, kmap = O.subdivide2(c)
    for shift in (0, 1):  # entries before the map: 0 is 16-byte aligned
        buf = s3dx.DeviceArray.from_host(np.full(8 * p * 27 + 8, 77, np.int32))
        rows = s3dx.DeviceArray((8 * p, 4), np.int32)
        s3dx.subdivide2(d, p, True, out=(rows, buf.ptr + 4 * shift))
        print(f"subdivide p={p} shift={shift}", flush=True)
        got = buf.download()
        assert np.array_equal(rows.download(), child)
        assert np.array_equal(got[shift:shift + 8 * p * 27].reshape(-1, 27), kmap)
        assert np.all(got[:shift] == 77) and np.all(got[shift + 8 * p * 27:] == 77)
    rows, none = s3dx.subdivide2(d, p, False)
    assert none is None and np.array_equal(rows.download(), child)


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 20011])
def test_coarsen_blocks(s3dx, O, n, ordered):
    c = _set(n, n, ordered)
    got = s3dx.coarsen2(s3dx.DeviceArray.from_host(c), n)
    want = O.coarsen2(c)
    print(f"coarsen n={n} ordered={ordered} nc={got[0]}", flush=True)
    nc = want[0]
    assert got[0] == nc
    assert np.array_equal(got[1].download()[:nc], want[1])
    assert np.array_equal(got[2].download(), want[2])
    assert np.array_equal(got[3].download()[:8 * nc], want[3])
    assert np.array_equal(got[4].download()[:nc].view(np.uint32), want[4].view(np.uint32))
