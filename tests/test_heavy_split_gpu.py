"""GPU parity of heavy rows that are split by columns over several workgroups, and of the wavefront-wise product loop.

A row of the heavy bin with more products than an eighth of a compute unit's share (at least 8192) is cut into column
ranges, each found in the B rows by binary search. Cases: one giant row among small ones (its products dwarf the rest), 40 rows
just over and under the smallest part size, rows of more than 1024 A entries (staged in chunks), B rows of 0, 1, 2, 63, 64, 65 and
thousands of entries next to each other, all products in a few columns (ranges that come out empty), a tile 2^19 columns wide and
one of 200 columns (one range only), and B rows whose columns are not sorted (the row then runs whole). Through
the two-phase call, the batched exact stage and the batched learned stage. Structure must equal the oracle's
(bcl/containers/algorithms/spgemm.hpp:40-76), values be within one rounding of the float64 oracle.
"""
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


def heavy_product(kind, n, dtype):
    rng = np.random.default_rng(5)
    lens = [0, 1, 2, 63, 64, 65, 7, min(n, 3000)] * 200  # B row lengths, repeated
    if kind == "few_columns":
        pool = np.sort(rng.choice(n, min(n, 3000), replace=False)) if n < 4096 else np.arange(n - 3000, n)
        brows = [np.sort(rng.choice(pool, min(x, pool.size), replace=False)) for x in lens]
    else:
        brows = [np.sort(rng.choice(n, x, replace=False)) for x in lens]
    k = len(brows)
    pick = lambda c: np.sort(rng.choice(k, c, replace=False))
    long_rows = np.flatnonzero(np.asarray(lens) == min(n, 3000))
    arows = [pick(3) for _ in range(50)]
    arows.append(pick(1500))  # giant: more than 1024 entries
    arows.append(np.arange(k))
    for c in (2, 3, 4, 20):  # 6000 to 60000 products
        arows += [np.sort(rng.choice(long_rows, c, replace=False)) for _ in range(10)]
    arows += [pick(30) for _ in range(20)] + [[]]
    return _csr(arows, k, rng, dtype), _csr(brows, n, rng, dtype)


def _check(c, ref, c64, bound, what):
    np.testing.assert_array_equal(c.row_ptr, ref.row_ptr, err_msg=what)
    np.testing.assert_array_equal(c.col_idx, ref.col_idx, err_msg=what)
    assert (np.abs(c.vals.astype(np.float64) - c64.vals) <= bound).all(), what


@pytest.mark.parametrize("kind,n,f64,ptr64", [("spread", 30000, False, False), ("spread", 1 << 19, True, True),
                                              ("few_columns", 1 << 19, False, True), ("spread", 200, True, False)])
def test_split_rows(handle, kind, n, f64, ptr64):
    dtype = np.float64 if f64 else np.float32
    a, b = heavy_product(kind, n, dtype)
    pd = torch.int64 if ptr64 else torch.int32
    A, B = DeviceCSR.from_host(a, ptr_dtype=pd), DeviceCSR.from_host(b, ptr_dtype=pd)
    ref, c64 = O.spgemm(a, b), O.spgemm_f64(a, b)
    pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, b)]
    bound = spgemm_value_bound(a, b, c64.vals, O.spgemm_f64(*pos).vals, dtype)
    print(f"[split] {kind} n={n} nnz={ref.nnz} two-phase", flush=True)
    _check(spgemm(handle, A, B, ptr_dtype=pd).to_host(), ref, c64, bound, "two-phase")
    tun, margin, slack = autotune.load_tuning()
    for mode in (BATCHED_EXACT, LEARNED):
        print(f"[split] stage mode {mode}", flush=True)
        plan = StagePlan(handle, [A, A], [B, B], mode=mode, params=predictor.load(), margin=margin, slack=slack, tuning=tun)
        plan.execute()
        torch.cuda.synchronize()
        for p in range(2):
            _check(plan.result_host(p), ref, c64, bound, f"stage mode {mode} product {p}")
        plan.close()


def test_unsorted_b_rows(handle):
    """B rows in random column order and one giant row whose output fits one LDS slice: same result as sorted."""
    rng = np.random.default_rng(9)
    n = 4096
    brows = [rng.permutation(rng.choice(n, 400, replace=False)) for _ in range(1300)]
    b = _csr(brows, n, rng, np.float32)
    order = np.concatenate([b.row_ptr[r] + np.argsort(b.col_idx[b.row_ptr[r]:b.row_ptr[r + 1]])
                            for r in range(b.m)]).astype(np.int64)
    sorted_b = CSR(b.m, n, b.row_ptr, b.col_idx[order], b.vals[order])
    a = _csr([np.arange(1300), np.arange(0, 1300, 2), np.arange(30), []], 1300, rng, np.float32)
    ref, c64 = O.spgemm(a, sorted_b), O.spgemm_f64(a, sorted_b)
    pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, sorted_b)]
    bound = spgemm_value_bound(a, sorted_b, c64.vals, O.spgemm_f64(*pos).vals, np.float32)
    _check(spgemm(handle, DeviceCSR.from_host(a), DeviceCSR.from_host(b)).to_host(), ref, c64, bound, "unsorted B")
