"""Calls on one handle across bclx_set_stream: a dense product returns while it runs, with its packed operands or its partial
sums in the handle's memory, and calls on the next stream must leave them alone. Results are compared bit for bit with
the same calls on one stream. A handle with a caller's allocator keeps nothing of a sum or a split."""
import ctypes

import pytest
import torch

from bcl_amd import gen
from bcl_amd._lib import call
from bcl_amd.device import (GEMM_BF16, GEMM_FP32, GEMM_SPLIT_BF16, DeviceCSR, Handle, accumulate, gemm, gemm_f64,
                            split_grid)
from test_failure_gpu import _HipAllocator

pytestmark = pytest.mark.gpu


def on(h, stream):
    call("bclx_set_stream", h.h, ctypes.c_void_p(stream.cuda_stream))


# packed operands in three arithmetics; partial sums of a product with few tiles and a long K (fp32, fp64)
PRODUCTS = [(4096, 4096, 4096, GEMM_FP32), (4096, 4096, 4096, GEMM_BF16), (3000, 2500, 4000, GEMM_SPLIT_BF16),
            (200, 100, 200000, GEMM_FP32), (200, 100, 200000, None)]


@pytest.mark.parametrize("m,n,k,mode", PRODUCTS)
def test_product_keeps_its_operands_across_streams(m, n, k, mode):
    dt = torch.float64 if mode is None else torch.float32
    g = torch.Generator(device="cuda").manual_seed(m + n)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dt)
    a, b, b2 = rand(m, k), rand(k, n), rand(k, n)
    csr = DeviceCSR.from_host(gen.rmat(13, seed=3))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    h = Handle(0, s1)

    def product(x):
        c = torch.zeros(m, n, dtype=dt, device="cuda")
        torch.cuda.synchronize()
        if mode is None:
            return gemm_f64(h, a, x, c)
        return gemm(h, a, x, c, mode=mode)

    want, want2 = product(b), product(b2)
    tiles = split_grid(h, csr, csr.m // 2, csr.n // 2)
    total = accumulate(h, [csr, csr])
    torch.cuda.synchronize()
    print(f"[streams] {m}x{n}x{k} mode {mode}", flush=True)
    c2 = torch.zeros(m, n, dtype=dt, device="cuda")
    for turn in range(3):
        on(h, s1)
        c1 = product(b)
        on(h, s2)
        if turn == 0:
            got = split_grid(h, csr, csr.m // 2, csr.n // 2)
            for key, t in got.items():
                assert torch.equal(t.row_ptr, tiles[key].row_ptr) and torch.equal(t.col_idx, tiles[key].col_idx)
                assert torch.equal(t.vals, tiles[key].vals)
        elif turn == 1:
            got = accumulate(h, [csr, csr])
            assert torch.equal(got.row_ptr, total.row_ptr) and torch.equal(got.col_idx, total.col_idx)
            assert torch.equal(got.vals, total.vals)
        else:
            (gemm_f64(h, a, b2, c2) if mode is None else gemm(h, a, b2, c2, mode=mode))
            torch.cuda.synchronize()
            assert torch.equal(c2, want2)
        torch.cuda.synchronize()
        assert torch.equal(c1, want), f"turn {turn}"
    h.close()


def test_captured_product_replays_after_a_stream_switch():
    g = torch.Generator(device="cuda").manual_seed(7)
    a, b = (torch.randn(700, 700, generator=g, device="cuda") for _ in range(2))
    c, want, other = (torch.zeros(700, 700, device="cuda") for _ in range(3))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    h = Handle(0, s1)
    torch.cuda.synchronize()
    gemm(h, a, b, want, mode=GEMM_SPLIT_BF16, beta=0.0)  # also makes the scratch, before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s1):
        gemm(h, a, b, c, mode=GEMM_SPLIT_BF16, beta=0.0)
    on(h, s2)
    for _ in range(3):
        gemm(h, a, b, other, mode=GEMM_SPLIT_BF16, beta=0.0)
        torch.cuda.synchronize()
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want) and torch.equal(other, want)
    h.close()


def test_no_callers_memory_is_kept_by_sums_and_splits():
    csr = DeviceCSR.from_host(gen.rmat(12, seed=3))
    h, al = Handle(0), _HipAllocator()
    try:
        al.install(h)
        accumulate(h, [csr, csr])
        split_grid(h, csr, csr.m // 2, csr.n // 2)
        assert al.allocs > 0 and not al.live
    finally:
        call("bclx_set_allocator", h.h, None, None, None)
        h.close()
