"""bclx_spmm of some rows of a matrix: row_ptr is part of the matrix's own, so it starts above 0 and ends below nnz, and the
entries outside it belong to no row. Values and B are small integers, so products are exact in any order; the rows of
C beyond A's are not touched."""
import numpy as np
import pytest
import torch

from bcl_amd.device import DeviceCSR, spmm
from test_split_entries_gpu import rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r0,r1", [(0, 3000), (1, 3000), (0, 2999), (1500, 1600), (1502, 1503), (2990, 3000), (5, 9)])
@pytest.mark.parametrize("n,bt,ptr", [(1, torch.float32, torch.int32), (64, torch.float32, torch.int64),
                                      (70, torch.bfloat16, torch.int32), (33, torch.float64, torch.int64)])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_rows_of_a_matrix(handle, r0, r1, n, bt, ptr, beta):
    rng = np.random.default_rng(r0 + n)
    k = 8000
    lens = rng.integers(0, 12, 3000)
    lens[1500:1503], lens[2998:] = (4000, 0, 3000), 0
    a = rows_of(list(lens), k, 1, np.float64 if bt == torch.float64 else np.float32)
    a.vals[:] = rng.integers(1, 5, a.vals.size)
    d = DeviceCSR.from_host(a, ptr_dtype=ptr)
    part = DeviceCSR(r1 - r0, k, d.row_ptr[r0:r1 + 1], d.col_idx, d.vals)
    b = rng.integers(-4, 5, (k, n)).astype(np.float64)
    ct = torch.float64 if bt == torch.float64 else torch.float32
    c = rng.integers(-4, 5, (r1 - r0 + 20, n)).astype(np.float64)
    want = c.copy()
    want[:r1 - r0] *= beta
    e0, e1 = a.row_ptr[r0], a.row_ptr[r1]
    rows = np.repeat(np.arange(r1 - r0), np.diff(a.row_ptr[r0:r1 + 1]))
    np.add.at(want, rows, a.vals[e0:e1, None].astype(np.float64) * b[a.col_idx[e0:e1]])
    print(f"[spmm] rows {r0} to {r1}, {n} columns {bt} beta {beta}", flush=True)
    C = torch.from_numpy(c).to("cuda", ct)
    torch.cuda.synchronize()
    spmm(handle, part, torch.from_numpy(b).to("cuda", bt), C, beta=beta)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(C.cpu().double().numpy(), want)
