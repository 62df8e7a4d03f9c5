"""bclx_csr_split_grid of some rows of a matrix: row_ptr is part of the matrix's own and does not start at 0, col_idx and
vals are the matrix's. Tiles are copies, so they are compared bit for bit."""
import numpy as np
import pytest
import torch

from bcl_amd.csr import get_slice
from bcl_amd.device import DeviceCSR, split_grid
from test_split_entries_gpu import rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r0,r1", [(0, 900), (1, 900), (450, 900), (450, 451), (7, 8), (899, 900)])
@pytest.mark.parametrize("dtype,ptr", [(np.float32, torch.int32), (np.float64, torch.int64)])
def test_split_rows_of_a_matrix(handle, r0, r1, dtype, ptr):
    n = 20000
    lens = np.random.default_rng(2).integers(0, 40, 900)
    lens[[3, 449, 600]] = 0, 9000, 5000
    a = rows_of(list(lens), n, 900, dtype)
    d = DeviceCSR.from_host(a, ptr_dtype=ptr)
    part = DeviceCSR(r1 - r0, n, d.row_ptr[r0:r1 + 1], d.col_idx, d.vals)
    tm, tn = (r1 - r0 + 1) // 2, n // 3 + 1
    print(f"[split] rows {r0} to {r1} of {a.m}", flush=True)
    got = split_grid(handle, part, tm, tn, ptr_dtype=ptr)
    for (i, j), t in got.items():
        t, w = t.to_host(), get_slice(a, r0 + i * tm, min(r0 + (i + 1) * tm, r1), j * tn, (j + 1) * tn)
        np.testing.assert_array_equal(t.row_ptr, w.row_ptr)
        np.testing.assert_array_equal(t.col_idx, w.col_idx)
        np.testing.assert_array_equal(t.vals.view(np.uint8), np.ascontiguousarray(w.vals).view(np.uint8))
