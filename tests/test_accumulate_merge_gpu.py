"""The K-way merge of bclx_accumulate_tiles at its edges: rows just below, at and above the length at which a row is
cut into column pieces, rows of many pieces, empty rows and tiles, the smallest and largest number of tiles the merge
takes, one more than that, and tiles whose columns are not sorted or repeat (the general path).

Every value is the float64 sum of its tiles' values in tile order, rounded once, so results are compared bit for bit.
"""
import numpy as np
import pytest
import torch

from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, accumulate

pytestmark = pytest.mark.gpu


def tile(m, n, lens, rng, dtype):
    """m x n with lens[i] distinct columns in row i, clustered towards low columns in the long rows."""
    cols = []
    for i, k in enumerate(lens):
        p = rng.random(n) * (1.0 + (np.arange(n) > n // 3))
        cols.append(np.sort(np.argpartition(p, k - 1)[:k]) if k else np.zeros(0, np.int64))
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    col = np.concatenate(cols).astype(np.int32) if len(cols) else np.zeros(0, np.int32)
    return CSR(m, n, rp, col, rng.uniform(-1, 1, col.size).astype(dtype))


def expected(tiles):
    m, n = tiles[0].m, tiles[0].n
    s, seen = np.zeros((m, n)), np.zeros((m, n), bool)
    for t in tiles:
        rows = np.repeat(np.arange(m), np.diff(t.row_ptr))
        for r, c, v in zip(rows, t.col_idx, t.vals.astype(np.float64)) if not sorted_unique(t) else ():
            s[r, c] += v
        if sorted_unique(t):
            s[rows, t.col_idx] += t.vals.astype(np.float64)
        seen[rows, t.col_idx] = True
    rp = np.concatenate([[0], np.cumsum(seen.sum(1))])
    return rp, np.nonzero(seen)[1], s[seen].astype(tiles[0].vals.dtype)


def sorted_unique(t):
    d = np.diff(t.col_idx.astype(np.int64))
    first = t.row_ptr[1:-1]
    first = first[(first > 0) & (first < t.nnz)] - 1
    d[first] = 1
    return bool((d > 0).all())


def check(handle, tiles, ptr=torch.int64, out=torch.int64):
    c = accumulate(handle, [DeviceCSR.from_host(t, ptr_dtype=ptr) for t in tiles], ptr_dtype=out).to_host()
    rp, col, val = expected(tiles)
    np.testing.assert_array_equal(c.row_ptr, rp)
    np.testing.assert_array_equal(c.col_idx, col)
    np.testing.assert_array_equal(c.vals.view(np.uint8), val.view(np.uint8))


@pytest.mark.parametrize("lens", [
    [[1024], [0]], [[1025], [0]], [[1000], [24]], [[1000], [25]],                 # a row at the piece length
    [[0, 700, 1023, 1, 0], [0, 700, 1, 1, 0]],                                    # pieces of several rows
    [[3000, 5, 2999, 0, 2500, 1], [2000, 5, 3000, 1, 0, 0], [1, 1, 3000, 0, 999, 0]],  # rows of several pieces
    [[0] * 300 + [1] + [0] * 2000 + [1]] * 2,                                     # mostly empty rows
])
def test_row_lengths(handle, lens):
    rng = np.random.default_rng(len(lens[0]))
    print("[merge] rows", [x[:6] for x in lens], flush=True)
    check(handle, [tile(len(x), 3000, x, rng, np.float32) for x in lens])


@pytest.mark.parametrize("K,dtype,ptr", [(1, np.float32, torch.int32), (2, np.float64, torch.int64),
                                         (5, np.float64, torch.int32), (33, np.float32, torch.int64),
                                         (64, np.float32, torch.int32), (65, np.float32, torch.int32)])
def test_tile_counts(handle, K, dtype, ptr):
    rng = np.random.default_rng(K)
    print(f"[merge] K={K} {dtype.__name__}", flush=True)
    tiles = [tile(40, 700, rng.integers(0, 90, 40) * (rng.random(40) < 0.8), rng, dtype) for _ in range(K)]
    tiles[K // 2] = CSR.empty(40, 700, dtype) if K > 2 else tiles[K // 2]
    check(handle, tiles, ptr, ptr)


@pytest.mark.parametrize("what", ["reversed", "repeated", "long"])
def test_unsorted_tiles_keep_their_sum(handle, what):
    rng = np.random.default_rng(3)
    n = 3000
    lens = [20, 0, 2600 if what == "long" else 30, 11]
    a, b = tile(4, n, lens, rng, np.float64), tile(4, n, [5, 9, 40, 0], rng, np.float64)
    e0, e1 = a.row_ptr[2], a.row_ptr[3]
    if what == "repeated":
        a.col_idx[e0 + 7] = a.col_idx[e0 + 6]
    else:
        a.col_idx[e0:e1] = a.col_idx[e0:e1][::-1]
    assert not sorted_unique(a)
    print("[merge] unsorted", what, flush=True)
    c = accumulate(handle, [DeviceCSR.from_host(t) for t in (a, b)]).to_host()
    rp, col, val = expected([a, b])
    np.testing.assert_array_equal(c.row_ptr, rp)
    np.testing.assert_array_equal(c.col_idx, col)
    # the general path may add an entry's two or three values in another order: two more float64 roundings
    assert np.all(np.abs(c.vals - val) <= 4 * 2.0 ** -53 * 3)
