"""SpMM where rows meet the work split: rows of one entry, rows as long as a group's run and one longer, rows that cross
one and several blocks of entries, long stretches of empty rows, one row holding everything; widths from one column to
several slices, with and without a remainder; a fresh C (beta 0, over NaN), an updated one (beta 1) and a scaled one;
padded and unaligned B and C. Operands are small integers, so sums are exact in any order and results are compared for
equality."""
import numpy as np
import pytest
import torch

from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spmm

pytestmark = pytest.mark.gpu

ROWS = {
    "mixed": [1, 0, 128, 129, 64, 65, 8, 9, 2047, 0, 0, 2049, 1, 1, 1, 700, 5000, 3] + [2] * 300 + [0] * 900 + [513, 511],
    "singles": [1] * 5000,
    "one row": [0, 0, 9000, 0],
    "short": [3, 0, 7, 1],
    "many": [9] * 30000 + [0] * 700 + [40] * 30000,
}


def matrix(lens, k, dtype, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    nnz = int(rp[-1])
    col = rng.integers(0, k, nnz).astype(np.int32)
    return CSR(len(lens), k, rp, col, rng.integers(-3, 4, nnz).astype(dtype))


def padded(rows, cols, dtype, g, pad, shift):
    flat = torch.full((rows * (cols + pad) + shift,), float("nan"), device="cuda", dtype=dtype)
    x = flat[shift:].view(rows, cols + pad)[:, :cols]
    x.copy_(torch.randint(-2, 3, (rows, cols), generator=g, device="cuda"))
    return x


@pytest.mark.parametrize("name,b_dtype,n,ptr", [
    ("mixed", "f32", 1, 4), ("mixed", "f32", 3, 8), ("mixed", "f32", 4, 4), ("mixed", "f32", 7, 4), ("mixed", "f32", 15, 4),
    ("mixed", "f32", 33, 4), ("mixed", "f32", 130, 8), ("mixed", "bf16", 2, 4), ("mixed", "bf16", 5, 4),
    ("mixed", "bf16", 9, 8), ("mixed", "bf16", 61, 4), ("mixed", "bf16", 129, 4), ("mixed", "f64", 1, 4),
    ("mixed", "f64", 3, 4), ("mixed", "f64", 37, 8), ("singles", "f32", 20, 4), ("singles", "bf16", 20, 4),
    ("one row", "f32", 70, 4), ("one row", "f64", 2, 4), ("short", "f32", 64, 4), ("short", "bf16", 8, 8),
    ("many", "f32", 128, 4), ("many", "bf16", 100, 4), ("many", "f64", 64, 4),
])
def test_rows(handle, name, b_dtype, n, ptr):
    vt = np.float64 if b_dtype == "f64" else np.float32
    a = matrix(ROWS[name], 501, vt, n)
    A = DeviceCSR.from_host(a, ptr_dtype=torch.int64 if ptr == 8 else torch.int32)
    bt = {"f32": torch.float32, "bf16": torch.bfloat16, "f64": torch.float64}[b_dtype]
    ct = torch.float64 if b_dtype == "f64" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(n)
    print(f"[spmm] {name} {a.m} rows, {a.nnz} entries, {b_dtype} x {n}", flush=True)
    for pad, shift in ((0, 0), (3, 1)):
        B, C0 = padded(a.n, n, bt, g, pad, shift), padded(a.m, n, ct, g, pad, shift)
        rows = torch.repeat_interleave(torch.arange(a.m, device="cuda"),
                                       torch.from_numpy(np.diff(a.row_ptr)).cuda())
        prod = torch.zeros(a.m, n, device="cuda", dtype=torch.float64).index_add_(
            0, rows, A.vals.double()[:, None] * B.double()[A.col_idx.long()])
        for alpha, beta in ((1.0, 1.0), (2.0, 0.0), (1.0, -2.0)):
            C = torch.full((a.m * (n + pad) + shift,), float("nan"), device="cuda", dtype=ct)
            C = C[shift:].view(a.m, n + pad)[:, :n]
            if beta != 0:
                C.copy_(C0)
            spmm(handle, A, B, C, alpha=alpha, beta=beta)
            want = alpha * prod + (beta * C0.double() if beta != 0 else 0)
            assert torch.equal(C.double(), want), (pad, alpha, beta)
