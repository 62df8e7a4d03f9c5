"""The entry-parallel tile copy of bclx_csr_split_grid at its edges: a row longer than a copying workgroup's chunk of
4096 entries, more than a window (256) of empty rows in a row, tile columns that do not divide a 256-thread block and
the largest number of them, one-row tiles, a single entry. Tiles are copies, so they are compared bit for bit."""
import numpy as np
import pytest
import torch

from bcl_amd.csr import CSR, get_slice
from bcl_amd.device import DeviceCSR, split_grid

pytestmark = pytest.mark.gpu


def rows_of(lens, n, seed, dtype):
    rng = np.random.default_rng(seed)
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens] + [np.zeros(0, np.int64)])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    return CSR(len(lens), n, rp, col.astype(np.int32), rng.uniform(-1, 1, col.size).astype(dtype))


HUB = [3, 0, 9000, 4096, 1] + [0] * 600 + [5000, 7]


@pytest.mark.parametrize("lens,n,tm,tn,dtype,ptr", [
    (HUB, 9999, 100, 3333, np.float32, torch.int32),      # 3 tile columns
    (HUB, 9999, 607, 1430, np.float64, torch.int64),      # 7 tile columns, one tile row
    (HUB, 9999, 1, 9999, np.float32, torch.int32),        # one-row tiles
    ([5, 0, 255, 256, 257, 1], 1024, 4, 4, np.float32, torch.int64),  # 256 tile columns
    ([0] * 700 + [1], 50, 300, 20, np.float32, torch.int32),          # a single entry after empty rows
])
def test_split_edges(handle, lens, n, tm, tn, dtype, ptr):
    a = rows_of(lens, n, len(lens), dtype)
    print(f"[split] {a.m}x{a.n} nnz={a.nnz} tiles {tm}x{tn}", flush=True)
    got = split_grid(handle, DeviceCSR.from_host(a, ptr_dtype=ptr), tm, tn, ptr_dtype=ptr)
    for (i, j), t in got.items():
        t, w = t.to_host(), get_slice(a, i * tm, (i + 1) * tm, j * tn, (j + 1) * tn)
        np.testing.assert_array_equal(t.row_ptr, w.row_ptr)
        np.testing.assert_array_equal(t.col_idx, w.col_idx)
        np.testing.assert_array_equal(t.vals.view(np.uint8), np.ascontiguousarray(w.vals).view(np.uint8))
