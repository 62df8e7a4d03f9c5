"""C's row_ptr in the memory of an operand's arrays: the numeric pass reads them to its end, so row_ptr comes after it."""
import ctypes

import pytest
import torch

from bcl_amd import gen
from bcl_amd._lib import call
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spgemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", ["A.row_ptr", "B.row_ptr", "A.col_idx", "A.vals", "inside B.col_idx"])
@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("entry", ["two-phase", "noalloc"])
def test_row_ptr_over_an_operand(handle, which, f64, entry):
    x = gen.rmat(13, seed=8)
    a = CSR(x.m, x.n, x.row_ptr, x.col_idx, x.vals.astype("float64") if f64 else x.vals)
    pd = torch.int64 if f64 else torch.int32
    A, B = DeviceCSR.from_host(a, ptr_dtype=pd), DeviceCSR.from_host(a, ptr_dtype=pd)
    want = spgemm(handle, A, B, ptr_dtype=pd)
    torch.cuda.synchronize()
    m = a.m
    over = lambda x, skip=0: x[:x.numel() // 2 * 2].view(pd)[skip:skip + m + 1]
    rp = {"A.row_ptr": A.row_ptr, "B.row_ptr": B.row_ptr, "A.col_idx": over(A.col_idx), "A.vals": over(A.vals),
          "inside B.col_idx": over(B.col_idx, 64)}[which]
    C = DeviceCSR(m, a.n, rp, torch.zeros(want.nnz, dtype=torch.int32, device="cuda"),
                  torch.zeros(want.nnz, dtype=A.vals.dtype, device="cuda"))
    torch.cuda.synchronize()
    da, db, dc = A.desc(), B.desc(), C.desc()
    print(f"[row_ptr] {which} f64={f64} {entry}", flush=True)
    if entry == "noalloc":
        call("bclx_spgemm_noalloc", handle.h, ctypes.byref(da), ctypes.byref(db), ctypes.byref(dc))
    else:
        plan, nnz = ctypes.c_void_p(), ctypes.c_int64()
        call("bclx_spgemm_symbolic", handle.h, ctypes.byref(da), ctypes.byref(db), ctypes.byref(plan), ctypes.byref(nnz))
        call("bclx_spgemm_numeric", plan, ctypes.byref(dc))
        call("bclx_spgemm_plan_destroy", plan)
    torch.cuda.synchronize()
    assert torch.equal(C.row_ptr, want.row_ptr) and torch.equal(C.col_idx, want.col_idx)
    assert torch.allclose(C.vals, want.vals, rtol=2.0 ** -22, atol=1e-12)
