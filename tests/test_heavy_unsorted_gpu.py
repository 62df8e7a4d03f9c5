"""Heavy rows over B rows whose columns are not sorted: the parts and slices of a row find their shares of each B row by
binary search, and what a search misses must be noticed.

Rows of 300000 to 400000 products and more entries than one LDS slice holds, in each a few B rows with one pair of
neighbouring columns swapped (mostly inside one part of the row, some across a slice's end), of more and of fewer A entries
than are staged at a time; and B rows in random order through the stage pipelines. Structure must equal the oracle's on the
sorted B, values be within one rounding of the float64 oracle."""
import numpy as np
import pytest
import torch

import oracle_py as O
from bcl_amd import autotune, predictor
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spgemm
from bcl_amd.stage import BATCHED_EXACT, LEARNED, StagePlan
from conftest import spgemm_value_bound

pytestmark = pytest.mark.gpu


def _csr(rows, n, rng, dtype):
    rp = np.concatenate([[0], np.cumsum([len(x) for x in rows])]).astype(np.int64)
    col = np.concatenate([np.asarray(x, np.int64) for x in rows]).astype(np.int32)
    return CSR(len(rows), n, rp, col, rng.uniform(-1, 1, col.size).astype(dtype))


def _sorted(b):
    row = np.repeat(np.arange(b.m), np.diff(b.row_ptr))
    order = np.lexsort((b.col_idx, row))
    return CSR(b.m, b.n, b.row_ptr, b.col_idx[order], b.vals[order])


def _check_all(handle, a, b, dtype, modes=("two-phase", BATCHED_EXACT, LEARNED), ptr=torch.int32):
    sb = _sorted(b)
    ref, c64 = O.spgemm(a, sb), O.spgemm_f64(a, sb)
    pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, sb)]
    bound = spgemm_value_bound(a, sb, c64.vals, O.spgemm_f64(*pos).vals, dtype)
    A, B = DeviceCSR.from_host(a, ptr_dtype=ptr), DeviceCSR.from_host(b, ptr_dtype=ptr)
    tun, margin, slack = autotune.load_tuning()
    for mode in modes:
        print(f"[unsorted] {mode}: nnz {ref.nnz}", flush=True)
        if mode == "two-phase":
            c = spgemm(handle, A, B).to_host()
        else:
            plan = StagePlan(handle, [A], [B], mode=mode, params=predictor.load(), margin=margin, slack=slack, tuning=tun)
            plan.execute()
            torch.cuda.synchronize()
            c = plan.result_host(0)
            plan.close()
        np.testing.assert_array_equal(c.row_ptr, ref.row_ptr, err_msg=str(mode))
        np.testing.assert_array_equal(c.col_idx, ref.col_idx, err_msg=str(mode))
        off = np.abs(c.vals.astype(np.float64) - c64.vals) > bound
        assert not off.any(), f"{mode}: {off.sum()} values out of bound"


@pytest.mark.parametrize("entries,f64", [(2000, False), (900, False), (2000, True)])
def test_swapped_neighbours_in_split_rows(handle, entries, f64):
    """100 rows of the same products in all, so each is split into parts of about 20000 products and 13000 entries."""
    rng = np.random.default_rng(entries)
    n, dtype = 1 << 19, np.float64 if f64 else np.float32
    blen = 400000 // entries
    brows = [np.sort(rng.choice(n, blen, replace=False)) for _ in range(4000)]
    swapped = np.arange(0, 4000, 8)  # one pair of neighbours each
    for r in swapped:
        q = int(rng.integers(0, blen - 1))
        brows[r][[q, q + 1]] = brows[r][[q + 1, q]]
    plain = np.setdiff1d(np.arange(4000), swapped)
    arows = [np.sort(np.concatenate([rng.choice(plain, entries - 5, replace=False),
                                     rng.choice(swapped, 5, replace=False)])) for _ in range(100)]
    a, b = _csr(arows, 4000, rng, dtype), _csr(brows, n, rng, dtype)
    _check_all(handle, a, b, dtype, ptr=torch.int64 if f64 else torch.int32)


def test_shuffled_b_rows_in_every_pipeline(handle):
    """Split rows whose parts are refused run whole: in one slice, and in several with more A entries than are staged."""
    rng = np.random.default_rng(9)
    for n, entries in ((4096, 1300), (30000, 1300), (30000, 700)):
        brows = [rng.permutation(rng.choice(n, 400, replace=False)) for _ in range(1300)]
        arows = [np.arange(entries), np.arange(0, 1300, 2), np.arange(30), []]
        a, b = _csr(arows, 1300, rng, np.float32), _csr(brows, n, rng, np.float32)
        _check_all(handle, a, b, np.float32)
