"""The packed dense kernels' operand copies: whole 64 x 64 tiles of 16-byte aligned operands are read 16 bytes per lane,
tiles at ragged ends and operands with an odd leading dimension or a base off 16 bytes element by element. Products large
enough for the packed kernels, in all four transpositions. Operands are small integers, so every product and sum is exact
in every arithmetic mode and results are compared for equality."""
import pytest
import torch

from bcl_amd.device import GEMM_BF16, GEMM_FP32, GEMM_SPLIT_BF16, gemm
from test_gemm_direct_gpu import operand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,m,n,k", [(GEMM_FP32, 4096, 4096, 1056), (GEMM_BF16, 4096, 2048, 1600),
                                        (GEMM_BF16, 2111, 2049, 1601), (GEMM_SPLIT_BF16, 1984, 2050, 1602)])
def test_packed_operands(handle, mode, m, n, k):
    for ta in (False, True):
        for tb in (False, True):
            for pad, shift in ((0, 0), (4, 0), (3, 0), (4, 1)):
                print(f"[pack] mode {mode} {m} x {n} x {k} ta={ta} tb={tb} pad={pad} shift={shift}", flush=True)
                a = operand(*((k, m) if ta else (m, k)), 1, torch.float32, pad, shift)
                b = operand(*((n, k) if tb else (k, n)), 2, torch.float32, pad, shift)
                c = operand(m, n, 3, torch.float32)
                want = c.double() + (a.t() if ta else a).double() @ (b.t() if tb else b).double()
                gemm(handle, a, b, c, mode=mode, trans_a=ta, trans_b=tb)
                assert torch.equal(c.double(), want), (ta, tb, pad, shift)
