"""bclx_accumulate_tiles on rows made of sorted runs one after the other: a cut of such a row into column pieces gives
pieces of more entries than a workgroup merges, and the tile must take the general path whatever the other tiles hold
there. Values are small integers, so the sums are exact in any order."""
import numpy as np
import pytest
import torch

from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, accumulate

pytestmark = pytest.mark.gpu


def one_row(n, cols, seed, dtype=np.float32):
    cols = np.asarray(cols, np.int32)
    vals = np.random.default_rng(seed).integers(1, 9, cols.size).astype(dtype)
    return CSR(3, n, np.array([0, 0, cols.size, cols.size], np.int64), cols, vals)


@pytest.mark.parametrize("n,runs", [(200000, [(100000, 105000), (0, 5000)]), (8192, [(5000, 8000), (0, 5000)]),
                                    (6000, [(3400, 6000), (0, 2600)]), (6000, [(2305, 4610), (0, 2305)])])
@pytest.mark.parametrize("other", ["none", "empty", "few", "alike"])
def test_rows_of_sorted_runs(handle, n, runs, other):
    cols = np.concatenate([np.arange(a, b) for a, b in runs])
    tiles = [one_row(n, cols, 1)]
    if other != "none":
        tiles.append(one_row(n, {"empty": [], "few": [1, n - 1], "alike": cols}[other], 2))
    s = np.zeros(n)
    for t in tiles:
        np.add.at(s, t.col_idx, t.vals.astype(np.float64))
    print(f"[merge] runs {runs} of {n}, other tile {other}", flush=True)
    c = accumulate(handle, [DeviceCSR.from_host(t, ptr_dtype=torch.int64) for t in tiles]).to_host()
    want = np.flatnonzero(s)
    np.testing.assert_array_equal(c.row_ptr, [0, 0, want.size, want.size])
    np.testing.assert_array_equal(c.col_idx, want)
    np.testing.assert_array_equal(c.vals, s[want])
