"""The dense kernels at the edges of their tiles: one element, one row, one short of a tile of 64 and one over it, fewer
rows than a micro-tile in the last tile, K below, at and past a K tile, K deep enough to be split over blocks, operands
that start off any vector alignment, padded leading dimensions, C in A's place. Operands are small integers, so every
product and sum is exact in every arithmetic mode and results are compared for equality."""
import pytest
import torch

from bcl_amd.device import GEMM_BF16, GEMM_FP32, GEMM_SPLIT_BF16, gemm, gemm_f64

pytestmark = pytest.mark.gpu
MODES = {"f32": GEMM_FP32, "bf16": GEMM_BF16, "split": GEMM_SPLIT_BF16, "f64": None}


def operand(rows, cols, seed, dtype, pad=0, shift=0):
    """rows x cols integers in [-8, 8], leading dimension cols + pad, starting `shift` elements into its storage."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    flat = torch.full((rows * (cols + pad) + shift,), 1e6, device="cuda", dtype=dtype)
    x = flat[shift:].view(rows, cols + pad)[:, :cols]
    x.copy_(torch.randint(-8, 9, (rows, cols), generator=g, device="cuda"))
    return x


def product(handle, mode, a, b, c, ta, tb, alpha, beta):
    if mode == "f64":
        return gemm_f64(handle, a, b, c, trans_a=ta, trans_b=tb, alpha=alpha, beta=beta)
    return gemm(handle, a, b, c, mode=MODES[mode], trans_a=ta, trans_b=tb, alpha=alpha, beta=beta)


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 65, 2), (64, 64, 64), (63, 67, 65), (66, 129, 15), (130, 5, 17),
                                   (65, 2, 2049), (200, 190, 700)])
def test_edges(handle, mode, m, n, k):
    print(f"[gemm] {mode} {m} x {n} x {k}", flush=True)
    dt = torch.float64 if mode == "f64" else torch.float32
    for ta in (False, True):
        for tb in (False, True):
            for pad, shift, beta in ((0, 0, 0.0), (3, 1, 1.0)):
                a = operand(*((k, m) if ta else (m, k)), 1, dt, pad, shift)
                b = operand(*((n, k) if tb else (k, n)), 2, dt, pad, shift)
                c = operand(m, n, 3, dt, pad, shift)
                want = beta * c.double() + 2 * (a.t() if ta else a).double() @ (b.t() if tb else b).double()
                product(handle, mode, a, b, c, ta, tb, 2.0, beta)
                assert torch.equal(c.double(), want), (ta, tb, pad)


@pytest.mark.parametrize("mode", list(MODES))
def test_c_in_the_place_of_an_operand(handle, mode):
    dt = torch.float64 if mode == "f64" else torch.float32
    a, b = operand(300, 300, 4, dt), operand(300, 300, 5, dt)
    want = a.double() + a.double() @ b.double()
    print("[gemm] in place", mode, flush=True)
    product(handle, mode, a, b, a, False, False, 1.0, 1.0)
    assert torch.equal(a.double(), want)
