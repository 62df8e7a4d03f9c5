"""bclx_accumulate_tiles into the arrays of one of its tiles, which have room for the sum. Values are small integers, so the
sums are exact in any order."""
import ctypes

import numpy as np
import pytest
import torch

from bcl_amd._lib import bclx_csr, call
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, accumulate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,ptr", [(np.float32, torch.int32), (np.float64, torch.int64)])
@pytest.mark.parametrize("where", ["columns and values", "columns", "values", "all three"])
def test_sum_over_its_first_tile(handle, dtype, ptr, where):
    rng = np.random.default_rng(6)
    m, n = 3000, 40000
    tiles = []
    for t in range(3):
        lens = rng.integers(0, 20, m)
        lens[m // 2] = 6000  # cut into pieces
        col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.int32)
        rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        tiles.append(CSR(m, n, rp, col, rng.integers(1, 9, col.size).astype(dtype)))
    dev = [DeviceCSR.from_host(t, ptr_dtype=ptr) for t in tiles]
    want = accumulate(handle, dev, ptr_dtype=ptr)
    nnz, own = want.nnz, dev[0].nnz
    roomy = lambda x: torch.cat([x, torch.zeros(nnz - own, dtype=x.dtype, device=x.device)])
    col, val = roomy(dev[0].col_idx), roomy(dev[0].vals)
    dev[0].col_idx, dev[0].vals = col[:own], val[:own]
    C = DeviceCSR(m, n, dev[0].row_ptr if where == "all three" else torch.zeros_like(dev[0].row_ptr),
                  torch.zeros_like(col) if where == "values" else col,
                  torch.zeros_like(val) if where == "columns" else val)
    arr = (bclx_csr * 3)(*[d.desc() for d in dev])
    d = C.desc()
    torch.cuda.synchronize()
    print(f"[in place] {where} {dtype.__name__}", flush=True)
    call("bclx_accumulate_tiles", handle.h, 3, arr, ctypes.byref(d))
    assert d.nnz == nnz
    assert torch.equal(C.row_ptr, want.row_ptr)
    assert torch.equal(C.col_idx, want.col_idx) and torch.equal(C.vals, want.vals)
