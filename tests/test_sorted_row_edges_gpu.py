"""GPU parity of the sort-based rows at the edges of their sizes (128 to 512 products per wavefront, then 1024, 2048 and
4096 over two, four and eight wavefronts).

Rows one product below, at and above each size: all columns different, one run of equal columns as long as the row (it
crosses every lane and wavefront), two columns in turn, runs of 3 to 700 products with ends inside lanes and wavefronts, as one
A entry with a long B row, as as many A entries of one product, and with empty B rows between. Structure equals the oracle's
(bcl/containers/algorithms/spgemm.hpp:40-76); values are within one rounding of the float64 oracle.
"""
import numpy as np
import pytest
import torch

import oracle_py as O
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spgemm
from conftest import spgemm_value_bound

pytestmark = pytest.mark.gpu

SIZES = [s + d for s in (64, 128, 256, 512, 1024, 2048, 4096) for d in (-1, 0, 1)]


def edge_product(n, dtype):
    rng = np.random.default_rng(3)
    brows, arows = [], []

    def b_row(cols):
        brows.append(np.sort(np.asarray(cols, np.int64)))
        return len(brows) - 1

    empty = b_row([])
    for p in SIZES:
        arows.append([b_row(rng.choice(n, min(p, n), replace=False))])
        ones = [b_row([c]) for c in rng.choice(n, p, replace=True)]
        arows.append(ones)
        same = [b_row([n // 2]) for _ in range(p)]
        arows.append(same)
        arows.append([x for i in range(p) for x in ([b_row([n - 1 - i % 2])] + ([empty] if i % 7 == 0 else []))])
        row, left = [], p
        while left > 0:  # runs of a few lengths: k entries whose B rows share their columns
            k = int(min(left, rng.choice([3, 9, 65, 700])))
            row += [b_row([n // 3 + left]) for _ in range(k)]
            left -= k
        arows.append(row + [empty])

    def mk(rows, width):
        rp = np.concatenate([[0], np.cumsum([len(x) for x in rows])]).astype(np.int64)
        col = np.concatenate([np.asarray(x, np.int64) for x in rows]).astype(np.int32)
        return CSR(len(rows), width, rp, col, rng.uniform(-1, 1, col.size).astype(dtype))

    return mk([np.unique(x) for x in arows], len(brows)), mk(brows, n)


@pytest.mark.parametrize("n,dtype,ptr64", [(1 << 19, np.float32, False), (20000, np.float64, False),
                                           (20000, np.float32, True), (1 << 19, np.float64, True)])
def test_sorted_row_edges(handle, n, dtype, ptr64):
    a, b = edge_product(n, dtype)
    pd = torch.int64 if ptr64 else torch.int32
    c = spgemm(handle, DeviceCSR.from_host(a, ptr_dtype=pd), DeviceCSR.from_host(b, ptr_dtype=pd)).to_host()
    ref = O.spgemm(a, b)
    np.testing.assert_array_equal(c.row_ptr, ref.row_ptr)
    np.testing.assert_array_equal(c.col_idx, ref.col_idx)
    c64 = O.spgemm_f64(a, b)
    pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, b)]
    bound = spgemm_value_bound(a, b, c64.vals, O.spgemm_f64(*pos).vals, dtype)
    assert (np.abs(c.vals.astype(np.float64) - c64.vals) <= bound).all()
