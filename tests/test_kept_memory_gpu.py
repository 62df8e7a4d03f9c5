"""The memory a handle keeps between calls comes back to the device when the caller asks (bclx_set_allocator), and a plan
that exists keeps its own."""
import ctypes

import pytest
import torch

from bcl_amd._lib import call
from bcl_amd.device import DeviceCSR, Handle, accumulate, spgemm

pytestmark = pytest.mark.gpu
M = 6_000_000  # rows: 104 bytes of plan workspace each, 20 of a sum's


def test_kept_workspace_is_given_back():
    rp = torch.zeros(M + 1, dtype=torch.int32, device="cuda")
    rp[1:] = 1
    a = DeviceCSR(M, M, rp, torch.zeros(1, dtype=torch.int32, device="cuda"), torch.ones(1, device="cuda"))
    h = Handle(0)
    free = lambda: (torch.cuda.synchronize(), torch.cuda.mem_get_info()[0])[1]
    spgemm(h, a, a)
    accumulate(h, [a, a])
    kept = free()
    call("bclx_set_allocator", h.h, None, None, None)
    assert free() - kept >= 120 * M, "the workspaces of the plan and of the sum"
    # a plan's workspace stays with it
    d = a.desc()
    plan, nnz = ctypes.c_void_p(), ctypes.c_int64()
    call("bclx_spgemm_symbolic", h.h, ctypes.byref(d), ctypes.byref(d), ctypes.byref(plan), ctypes.byref(nnz))
    before = free()
    call("bclx_set_allocator", h.h, None, None, None)
    assert free() == before and nnz.value == 1
    c = DeviceCSR(M, M, torch.full_like(rp, -1), torch.full((1,), -1, dtype=torch.int32, device="cuda"),
                  torch.zeros(1, device="cuda"))
    dc = c.desc()
    call("bclx_spgemm_numeric", plan, ctypes.byref(dc))
    call("bclx_spgemm_plan_destroy", plan)
    torch.cuda.synchronize()
    assert torch.equal(c.row_ptr, rp) and int(c.col_idx) == 0 and float(c.vals) == 1.0
    h.close()
