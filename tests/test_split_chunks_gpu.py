"""The tile copy's chunks of 4096 entries plus rows and windows of 1024 rows at their edges: chunks of empty rows only, a
window more and a window less than a chunk of them, rows that end where a chunk does, a hub row over many chunks followed and
preceded by long empty stretches, one entry per row. Tiles are copies, so they are compared bit for bit."""
import numpy as np
import pytest
import torch

from bcl_amd.csr import get_slice
from bcl_amd.device import DeviceCSR, split_grid
from test_split_entries_gpu import rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [
    [0] * 9000 + [1],
    [1] * 9001,
    [0] * 1023 + [3073] + [0] * 1024 + [3072, 0, 4095, 4096, 1],  # rows ending on, before and after a chunk's weight
    [0] * 5000 + [20000] + [0] * 6000 + [2] * 3000 + [0] * 4095 + [5],
    [4095, 4095, 4095] + [0] * 4096 + [4094],
])
@pytest.mark.parametrize("dtype,ptr", [(np.float32, torch.int32), (np.float64, torch.int64)])
def test_split_chunks(handle, lens, dtype, ptr):
    n = 25000
    a = rows_of(lens, n, len(lens), dtype)
    tm, tn = (a.m + 2) // 3, n // 4 + 1
    print(f"[split] {a.m}x{a.n} nnz={a.nnz} tiles {tm}x{tn}", flush=True)
    got = split_grid(handle, DeviceCSR.from_host(a, ptr_dtype=ptr), tm, tn, ptr_dtype=ptr)
    for (i, j), t in got.items():
        t, w = t.to_host(), get_slice(a, i * tm, (i + 1) * tm, j * tn, (j + 1) * tn)
        np.testing.assert_array_equal(t.row_ptr, w.row_ptr)
        np.testing.assert_array_equal(t.col_idx, w.col_idx)
        np.testing.assert_array_equal(t.vals.view(np.uint8), np.ascontiguousarray(w.vals).view(np.uint8))
