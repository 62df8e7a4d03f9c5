"""GPU parity of the register-sorted rows at the edges of their two sizes (32 and 64 products per row).

Rows of exactly 1, 3, 4, 5, 8, 9, 31, 32, 33, 47, 63, 64 and 65 products (65 goes to the next kernel), each as products
that all differ in column, that all share one column (a run as long as the row) and that mix both, as one A entry with a
long B row, as many A entries of one product each, and with empty B rows between them. The row count leaves the last
wavefront partly filled. Structure equals the oracle's (bcl/containers/algorithms/spgemm.hpp:40-76); values are within
one rounding of the float64 oracle.
"""
import numpy as np
import pytest
import torch

import oracle_py as O
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spgemm
from conftest import spgemm_value_bound

pytestmark = pytest.mark.gpu

SIZES = (1, 3, 4, 5, 8, 9, 31, 32, 33, 47, 63, 64, 65)
N = 4096


def edge_product(dtype):
    rng = np.random.default_rng(11)
    brows, arows = [], []

    def b_row(cols):
        brows.append(np.sort(np.asarray(cols, np.int64)))
        return len(brows) - 1

    for rep in range(3):
        for p in SIZES:
            arows.append([b_row(rng.choice(N, p, replace=False))])  # one entry, all columns differ
            arows.append([b_row([N - 1 - rep]) for _ in range(p)])  # one run of p products
            distinct = rng.choice(N, p, replace=False)
            arows.append([b_row([c]) for c in distinct])  # p entries of one product, unsorted columns
            row, left = [], p  # repeated columns, with empty B rows between
            pool = rng.choice(N, 9, replace=False)
            while left > 0:
                k = int(min(left, rng.integers(1, 8)))
                row += [b_row(rng.choice(pool, k, replace=False)), b_row([])]
                left -= k
            arows.append(row)
            arows.append([])

    def mk(rows, n):
        rp = np.concatenate([[0], np.cumsum([len(x) for x in rows])]).astype(np.int64)
        col = np.concatenate([np.asarray(x, np.int64) for x in rows]).astype(np.int32)
        return CSR(len(rows), n, rp, col, rng.uniform(-1, 1, col.size).astype(dtype))

    return mk(arows, len(brows)), mk(brows, N)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ptr64", [False, True])
def test_small_row_edges(handle, dtype, ptr64):
    a, b = edge_product(dtype)
    pd = torch.int64 if ptr64 else torch.int32
    c = spgemm(handle, DeviceCSR.from_host(a, ptr_dtype=pd), DeviceCSR.from_host(b, ptr_dtype=pd)).to_host()
    ref = O.spgemm(a, b)
    np.testing.assert_array_equal(c.row_ptr, ref.row_ptr)
    np.testing.assert_array_equal(c.col_idx, ref.col_idx)
    c64 = O.spgemm_f64(a, b)
    pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, b)]
    bound = spgemm_value_bound(a, b, c64.vals, O.spgemm_f64(*pos).vals, dtype)
    assert (np.abs(c.vals.astype(np.float64) - c64.vals) <= bound).all()
