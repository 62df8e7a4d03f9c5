"""The calls that a program of this library spends its time in, as measurable cases.

Each case is one pass through a public entry point of bcl_amd (device.spgemm, device.spmm, device.gemm,
device.gemm_f64, device.accumulate, device.split_grid, stage.StagePlan) on inputs that are made on the GPU from a
seed. The matrices are the ones this library is written for: uniform random rows, R-MAT graphs (edge factor and
quadrant probabilities as in bcl_amd.gen), five-point stencils with varying coefficients, and dense tiles of
standard normal values.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from bcl_amd import autotune, predictor
from bcl_amd.csr import grid_tile_shape
from bcl_amd.device import (GEMM_BF16, GEMM_FP32, GEMM_SPLIT_BF16, DeviceCSR, Handle, accumulate, gemm, gemm_f64,
                            spgemm, split_grid, spmm)
from bcl_amd.stage import LEARNED, StagePlan

DEV = "cuda" if torch.cuda.is_available() else "cpu"
RMAT_ABC = (0.57, 0.19, 0.19)
DTYPES = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}
GEMM_MODES = {"f32": GEMM_FP32, "bf16": GEMM_BF16, "split": GEMM_SPLIT_BF16}
CHUNK = 1 << 25  # products (or gathered values) expanded at a time by the 64-bit references

_handle = None


def handle() -> Handle:
    """The program's handle: one for all its calls."""
    global _handle
    if _handle is None:
        _handle = Handle(0)
    return _handle


def listed():
    return [
        # a small local block: what a fine-grained tile of an SPMatrix multiplies; launches and host work count
        {"name": "spgemm_small", "kind": "spgemm", "matrix": "uniform", "m": 500, "k": 500, "n": 500, "per_row": 6,
         "square": True, "dtype": "f32", "ptr": 4},
        # the benchmark's single tile: 16384^2 with 8 entries per row, C = A * A
        {"name": "spgemm_uniform", "kind": "spgemm", "matrix": "uniform", "m": 16384, "k": 16384, "n": 16384,
         "per_row": 8, "square": True, "dtype": "f32", "ptr": 4},
        # a whole graph squared on one GPU: rows from a few products to hubs of hundreds of thousands
        {"name": "spgemm_rmat", "kind": "spgemm", "matrix": "rmat", "scale": 16, "ef": 8, "square": True,
         "dtype": "f32", "ptr": 4},
        # the benchmark's FP64 stencil square: 16.7 M short rows on a 16.7 M-column tile
        {"name": "spgemm_stencil_f64", "kind": "spgemm", "matrix": "stencil", "grid": 4096, "square": True,
         "dtype": "f64", "ptr": 4},
        # a planned SUMMA stage replayed with its results handed out: 16 uneven products on 524288^2 tiles
        {"name": "stage_rmat", "kind": "stage", "scale": 21, "ef": 16, "grid": 4, "k": 3},
        # the benchmark's SpMM: a graph times 128 dense columns, added to C as BCL's spmm_wrapper does
        {"name": "spmm_f32", "kind": "spmm", "matrix": "rmat", "scale": 20, "ef": 16, "cols": 128, "b": "f32",
         "beta": 1.0, "ptr": 4},
        # feature aggregation: bf16 features, a width that is no power of two, C written anew
        {"name": "spmm_bf16", "kind": "spmm", "matrix": "rmat", "scale": 18, "ef": 16, "cols": 100, "b": "bf16",
         "beta": 0.0, "ptr": 4},
        # the benchmark's large dense tile in bf16
        {"name": "gemm_bf16", "kind": "gemm", "mode": "bf16", "m": 8192, "n": 8192, "k": 8192, "ta": False,
         "tb": False, "beta": 0.0},
        # an ordinary fp32 tile with ragged sides, added to C as BCL's gemm does
        {"name": "gemm_f32", "kind": "gemm", "mode": "f32", "m": 2000, "n": 1500, "k": 3001, "ta": False, "tb": True,
         "beta": 1.0},
        # the double overload on a ragged tile, A transposed
        {"name": "gemm_f64", "kind": "gemm", "mode": "f64", "m": 1234, "n": 2048, "k": 1777, "ta": True, "tb": False,
         "beta": 1.0},
        # the sum of a C tile's partial products over eight stages
        {"name": "accumulate", "kind": "accumulate", "tiles": 8, "scale": 16, "ef": 24, "dtype": "f32", "ptr": 8},
        # ingest: a graph in HBM cut into its tile grid
        {"name": "split_grid", "kind": "split", "matrix": "rmat", "scale": 20, "ef": 16, "gm": 4, "gn": 4,
         "dtype": "f32", "ptr": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(rng, v):
    """About half of the sizes off any power of two."""
    return max(1, v - rng.randrange(0, 8)) if rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["spgemm", "spgemm", "spmm", "spmm", "gemm", "gemm", "accumulate", "split", "stage"])
    if kind == "spgemm":
        what = rng.choice(["uniform", "uniform", "rmat", "stencil"])
        dtype, ptr = rng.choice(["f32", "f32", "f64"]), rng.choice([4, 8])
        if what == "uniform":
            m = _odd(rng, _log_int(rng, 64, 200000))
            square = rng.random() < 0.5
            k = m if square else _odd(rng, _log_int(rng, 64, 200000))
            n = m if square else _odd(rng, _log_int(rng, 64, 200000))
            return {"kind": kind, "matrix": what, "m": m, "k": k, "n": n, "per_row": rng.randrange(1, 17),
                    "square": square, "dtype": dtype, "ptr": ptr}
        if what == "rmat":
            return {"kind": kind, "matrix": what, "scale": rng.randrange(9, 16), "ef": rng.randrange(3, 13),
                    "square": True, "dtype": dtype, "ptr": ptr}
        return {"kind": kind, "matrix": what, "grid": _log_int(rng, 20, 3000), "square": True, "dtype": dtype,
                "ptr": ptr}
    if kind == "spmm":
        c = {"kind": kind, "cols": _log_int(rng, 1, 256), "b": rng.choice(["f32", "bf16", "f64"]),
             "beta": rng.choice([0.0, 1.0]), "ptr": rng.choice([4, 8])}
        if rng.random() < 0.5:
            c.update({"matrix": "rmat", "scale": rng.randrange(10, 19), "ef": rng.randrange(4, 17)})
        else:
            c.update({"matrix": "uniform", "m": _odd(rng, _log_int(rng, 100, 500000)),
                      "k": _odd(rng, _log_int(rng, 100, 500000)), "per_row": rng.randrange(1, 33)})
        return c
    if kind == "gemm":
        mode = rng.choice(["f32", "bf16", "split", "f64"])
        top = 8192 if mode in ("bf16", "split") else 4096
        m, n, k = (_odd(rng, _log_int(rng, 64, top)) for _ in range(3))
        return {"kind": kind, "mode": mode, "m": m, "n": n, "k": k, "ta": rng.random() < 0.5,
                "tb": rng.random() < 0.5, "beta": rng.choice([0.0, 1.0])}
    if kind == "accumulate":
        return {"kind": kind, "tiles": rng.randrange(2, 11), "scale": rng.randrange(8, 17), "ef": rng.randrange(2, 25),
                "dtype": rng.choice(["f32", "f32", "f64"]), "ptr": rng.choice([4, 8])}
    if kind == "split":
        gm, gn = rng.randrange(1, 5), rng.randrange(1, 5)
        dtype, ptr = rng.choice(["f32", "f32", "f64"]), rng.choice([4, 8])
        if rng.random() < 0.5:
            return {"kind": kind, "matrix": "rmat", "scale": rng.randrange(10, 20), "ef": rng.randrange(4, 17),
                    "gm": gm, "gn": gn, "dtype": dtype, "ptr": ptr}
        return {"kind": kind, "matrix": "uniform", "m": _odd(rng, _log_int(rng, 100, 1000000)),
                "k": _odd(rng, _log_int(rng, 100, 1000000)), "per_row": rng.randrange(1, 33), "gm": gm, "gn": gn,
                "dtype": dtype, "ptr": ptr}
    grid = rng.choice([2, 3, 4])
    scale = rng.randrange(12, {2: 18, 3: 20, 4: 21}[grid])
    return {"kind": "stage", "scale": scale, "ef": rng.randrange(8, 17), "grid": grid, "k": grid - 1}


# ---- inputs: plain CSR matrices (m, n, row_ptr int64, col int32, vals) on the GPU -----------------------------
# A matrix's pattern is drawn once for its sizes and then rotated (row and column numbers move on by a shift that
# the seed gives, within each tile where the matrix is cut into tiles), so that every seed gives another matrix
# with as many entries, and its product as many too. Values come from the seed alone.


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 11)


def _shift(seed):
    return int(np.random.RandomState(int(seed) % (1 << 31)).randint(0, 1 << 20))


def _rotated(i, size, block, shift):
    """i moved on by shift within its block of the dimension (the last block may be shorter)."""
    start = torch.div(i, block, rounding_mode="floor") * block
    length = torch.clamp(size - start, max=block)
    return start + (i - start + shift) % length


def _from_entries(row, col, m, n, seed, g, dtype, blocks):
    """The CSR matrix of the distinct entries, rotated within blocks, with values uniform in [-1, 1)."""
    s = _shift(seed)
    keys = torch.unique(_rotated(row, m, blocks[0], s) * n + _rotated(col, n, blocks[1], s))
    row = torch.div(keys, n, rounding_mode="floor")
    rp = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(torch.bincount(row, minlength=m), 0)
    vals = torch.rand(keys.numel(), generator=g, device=DEV, dtype=torch.float32) * 2 - 1
    return m, n, rp, (keys - row * n).to(torch.int32), vals.to(dtype)


def _uniform(m, n, per_row, seed, g, dtype, blocks=None):
    pattern = _generator(m * 31 + n * 17 + per_row)
    col = torch.randint(0, n, (m, per_row), generator=pattern, device=DEV)
    row = torch.arange(m, device=DEV)[:, None].expand(m, per_row)
    return _from_entries(row.reshape(-1), col.reshape(-1), m, n, seed, g, dtype, blocks or (m, n))


def _rmat(scale, ef, seed, g, dtype, blocks=None, which=0):
    pattern = _generator(scale * 31 + ef * 1009 + which)
    edges = ef << scale
    a, b, c = RMAT_ABC
    row = torch.zeros(edges, dtype=torch.int64, device=DEV)
    col = torch.zeros(edges, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        u = torch.rand(edges, generator=pattern, device=DEV)
        row = row * 2 + (u >= a + b)
        col = col * 2 + (((u >= a) & (u < a + b)) | (u >= a + b + c))
    n = 1 << scale
    return _from_entries(row, col, n, n, seed, g, dtype, blocks or (n, n))


def _stencil(grid, g, dtype):
    """Five-point stencil on a grid x grid mesh: neighbours -1 +- 0.2, diagonal 4 +- 0.2."""
    n = grid * grid
    i = torch.arange(n, device=DEV)
    x, y = i % grid, i // grid
    col = torch.stack([i - grid, i - 1, i, i + 1, i + grid], 1)
    keep = torch.stack([y > 0, x > 0, torch.ones_like(x, dtype=torch.bool), x < grid - 1, y < grid - 1], 1)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(keep.sum(1), 0)
    vals = torch.rand((n, 5), generator=g, device=DEV, dtype=torch.float32) * 0.4 - 1.2
    vals[:, 2] += 5.0
    return n, n, rp, col[keep].to(torch.int32), vals[keep].to(dtype)


def _matrix(case, seed, g, dtype, blocks=None):
    if case["matrix"] == "uniform":
        return _uniform(case["m"], case["k"], case["per_row"], seed, g, dtype, blocks)
    if case["matrix"] == "rmat":
        return _rmat(case["scale"], case["ef"], seed, g, dtype, blocks)
    return _stencil(case["grid"], g, dtype)


def _device(a, ptr):
    m, n, rp, col, vals = a
    return DeviceCSR(m, n, rp if ptr == 8 else rp.to(torch.int32), col, vals)


def _spgemm_inputs(case, seed):
    g, dtype = _generator(seed), DTYPES[case["dtype"]]
    a = _matrix(case, seed, g, dtype)
    b = a if case["square"] else _uniform(case["k"], case["n"], case["per_row"], seed, g, dtype)
    return a, b


def _spmm_inputs(case, seed):
    g = _generator(seed)
    ct = torch.float64 if case["b"] == "f64" else torch.float32
    a = _matrix(case, seed, g, ct)
    b = torch.randn((a[1], case["cols"]), generator=g, device=DEV, dtype=ct).to(DTYPES[case["b"]])
    return a, b, torch.randn((a[0], case["cols"]), generator=g, device=DEV, dtype=ct)


def _gemm_inputs(case, seed):
    g = _generator(seed)
    dt = torch.float64 if case["mode"] == "f64" else torch.float32
    m, n, k = case["m"], case["n"], case["k"]
    a = torch.randn((k, m) if case["ta"] else (m, k), generator=g, device=DEV, dtype=dt)
    b = torch.randn((n, k) if case["tb"] else (k, n), generator=g, device=DEV, dtype=dt)
    return a, b, torch.randn((m, n), generator=g, device=DEV, dtype=dt)


def _accumulate_inputs(case, seed):
    g = _generator(seed)
    return [_rmat(case["scale"], case["ef"], seed, g, DTYPES[case["dtype"]], which=t) for t in range(case["tiles"])]


def _split_input(case, seed):
    """The matrix to cut and its tile shape."""
    m, n = (case["m"], case["k"]) if case["matrix"] == "uniform" else (1 << case["scale"],) * 2
    shape = grid_tile_shape(m, n, case["gm"], case["gn"])
    return _matrix(case, seed, _generator(seed), DTYPES[case["dtype"]], shape), shape


def _stage_input(case, seed):
    """The matrix of a stage and its tile shape."""
    n = 1 << case["scale"]
    shape = grid_tile_shape(n, n, case["grid"], case["grid"])
    return _rmat(case["scale"], case["ef"], seed, _generator(seed), torch.float32, shape), shape


def prepare(case, seed):
    kind = case["kind"]
    if kind == "spgemm":
        a, b = _spgemm_inputs(case, seed)
        A = _device(a, case["ptr"])
        return {"kind": kind, "A": A, "B": A if b is a else _device(b, case["ptr"])}
    if kind == "spmm":
        a, b, c = _spmm_inputs(case, seed)
        return {"kind": kind, "A": _device(a, case["ptr"]), "B": b, "C": c, "beta": case["beta"]}
    if kind == "gemm":
        a, b, c = _gemm_inputs(case, seed)
        return {"kind": kind, "A": a, "B": b, "C": c, "mode": case["mode"], "ta": case["ta"], "tb": case["tb"],
                "beta": case["beta"]}
    if kind == "accumulate":
        return {"kind": kind, "tiles": [_device(t, case["ptr"]) for t in _accumulate_inputs(case, seed)]}
    if kind == "split":
        a, (tm, tn) = _split_input(case, seed)
        return {"kind": kind, "A": _device(a, case["ptr"]), "tm": tm, "tn": tn}
    # a stage: the tiles cut on the GPU, the plan made once for their structure
    a, (tm, tn) = _stage_input(case, seed)
    grid, k = case["grid"], case["k"]
    tiles = split_grid(handle(), _device(a, 4), tm, tn)
    tuning, margin, slack = autotune.load_tuning()
    plan = StagePlan(handle(), [tiles[(i, k)] for i in range(grid) for _ in range(grid)],
                     [tiles[(k, j)] for _ in range(grid) for j in range(grid)], mode=LEARNED,
                     params=predictor.load(), margin=margin, slack=slack, tuning=tuning)
    return {"kind": "stage", "plan": plan}


class _PlanArray:
    """A plan's device array as torch reads it without a copy; keeps the plan alive."""

    def __init__(self, plan, ptr, count, typestr):
        self.plan = plan
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _plan_tensor(plan, ptr, count, typestr, dtype):
    if count == 0:
        return torch.empty(0, dtype=dtype, device=DEV)
    return torch.as_tensor(_PlanArray(plan, ptr, count, typestr), device=DEV)


def run(state):
    kind, h = state["kind"], handle()
    if kind == "spgemm":
        c = spgemm(h, state["A"], state["B"])
        return c.row_ptr, c.col_idx, c.vals
    if kind == "spmm":
        return spmm(h, state["A"], state["B"], state["C"], beta=state["beta"])
    if kind == "gemm":
        a, b, c = state["A"], state["B"], state["C"]
        if state["mode"] == "f64":
            return gemm_f64(h, a, b, c, trans_a=state["ta"], trans_b=state["tb"], beta=state["beta"])
        return gemm(h, a, b, c, mode=GEMM_MODES[state["mode"]], trans_a=state["ta"], trans_b=state["tb"],
                    beta=state["beta"])
    if kind == "accumulate":
        c = accumulate(h, state["tiles"])
        return c.row_ptr, c.col_idx, c.vals
    if kind == "split":
        tiles = split_grid(h, state["A"], state["tm"], state["tn"])
        return [(t.row_ptr, t.col_idx, t.vals) for _, t in sorted(tiles.items())]
    plan = state["plan"]
    plan.execute()
    out = []
    for p in range(plan.npairs):
        d = plan.result_desc(p)
        out.append((_plan_tensor(plan, d.row_ptr, d.m + 1, "<i8", torch.int64),
                    _plan_tensor(plan, d.col_idx, d.nnz, "<i4", torch.int32),
                    _plan_tensor(plan, d.vals, d.nnz, "<f4", torch.float32)))
    return out


# ---- references in 64 bits, plain torch -------------------------------------------------------------------------


def _product_chunks(a, b, want_values):
    """C = A * B a group of whole rows at a time: (keys row * n + column, sorted and distinct; float64 sums)."""
    m, _, arp, acol, aval = a
    n, brp, bcol, bval = b[1], b[2], b[3], b[4]
    blen = brp[1:] - brp[:-1]
    per = blen[acol.long()]
    cum = torch.zeros(per.numel() + 1, dtype=torch.int64, device=per.device)
    cum[1:] = torch.cumsum(per, 0)
    row_end = cum[arp].cpu().numpy()
    arp_h = arp.cpu().numpy()
    rows = torch.repeat_interleave(torch.arange(m, device=per.device), arp[1:] - arp[:-1])
    r0 = 0
    while r0 < m:
        r1 = int(np.searchsorted(row_end, row_end[r0] + CHUNK, side="right")) - 1
        r1 = min(m, max(r0 + 1, r1))
        e0, e1, total = int(arp_h[r0]), int(arp_h[r1]), int(row_end[r1] - row_end[r0])
        r0 = r1
        if total == 0:
            continue
        e = torch.repeat_interleave(torch.arange(e0, e1, device=per.device), per[e0:e1], output_size=total)
        q = brp[acol[e].long()] + torch.arange(total, device=per.device) + cum[e0] - cum[e]
        key = rows[e] * n + bcol[q].long()
        if want_values:
            keys, inv = torch.unique(key, return_inverse=True)
            v = aval[e].double() * bval[q].double()
            yield keys, torch.zeros(keys.numel(), dtype=torch.float64, device=v.device).index_add_(0, inv, v)
        else:
            yield torch.unique(key), None


def _csr_of_keys(keys, m, n):
    row = torch.div(keys, n, rounding_mode="floor")
    rp = torch.zeros(m + 1, dtype=torch.int64, device=keys.device)
    rp[1:] = torch.cumsum(torch.bincount(row, minlength=m), 0)
    return rp, (keys - row * n).to(torch.int32)


def _cat(parts, dtype):
    return torch.cat(parts) if parts else torch.empty(0, dtype=dtype, device=DEV)


def _product64(a, b):
    ks, vs = [], []
    for k, v in _product_chunks(a, b, True):
        ks.append(k)
        vs.append(v)
    rp, col = _csr_of_keys(_cat(ks, torch.int64), a[0], b[1])
    return rp, col, _cat(vs, torch.float64)


def _product_size(a, b):
    """(products, entries) of C = A * B."""
    products = int((b[2][1:] - b[2][:-1])[a[3].long()].sum())
    return products, sum(k.numel() for k, _ in _product_chunks(a, b, False))


def _slice(a, r0, r1, c0, c1):
    """Rows [r0, r1), columns [c0, c1) of a matrix, columns shifted to start at 0."""
    _, _, rp, col, vals = a
    e0, e1 = int(rp[r0]), int(rp[r1])
    col, vals = col[e0:e1], vals[e0:e1]
    keep = (col >= c0) & (col < c1)
    before = torch.zeros(e1 - e0 + 1, dtype=torch.int64, device=col.device)
    before[1:] = torch.cumsum(keep, 0)
    return r1 - r0, c1 - c0, before[rp[r0:r1 + 1] - e0], col[keep] - c0, vals[keep]


def _grid(a, shape):
    tm, tn = shape
    rows = [(r, min(r + tm, a[0])) for r in range(0, a[0], tm)]
    cols = [(c, min(c + tn, a[1])) for c in range(0, a[1], tn)]
    return rows, cols


def _stage_operands(case, seed):
    a, shape = _stage_input(case, seed)
    rows, cols = _grid(a, shape)
    k = case["k"]
    return _slice(a, 0, a[0], *cols[k]), _slice(a, *rows[k], 0, a[1]), rows, cols


def exact(case, seed):
    kind = case["kind"]
    if kind == "spgemm":
        return _product64(*_spgemm_inputs(case, seed))
    if kind == "spmm":
        a, b, c = _spmm_inputs(case, seed)
        out = c.double() * case["beta"]
        rows = torch.repeat_interleave(torch.arange(a[0], device=DEV), a[2][1:] - a[2][:-1])
        step = max(1, CHUNK // max(1, case["cols"]))
        for e in range(0, rows.numel(), step):
            v = b[a[3][e:e + step].long()].double() * a[4][e:e + step, None].double()
            out.index_add_(0, rows[e:e + step], v)
        return out
    if kind == "gemm":
        a, b, c = _gemm_inputs(case, seed)
        a, b = a.double(), b.double()
        return c.double() * case["beta"] + (a.t() if case["ta"] else a) @ (b.t() if case["tb"] else b)
    if kind == "accumulate":
        tiles = _accumulate_inputs(case, seed)
        m, n = tiles[0][0], tiles[0][1]
        key = torch.cat([torch.repeat_interleave(torch.arange(m, device=DEV), t[2][1:] - t[2][:-1]) * n + t[3].long()
                         for t in tiles])
        keys, inv = torch.unique(key, return_inverse=True)
        v = torch.cat([t[4] for t in tiles]).double()
        rp, col = _csr_of_keys(keys, m, n)
        return rp, col, torch.zeros(keys.numel(), dtype=torch.float64, device=DEV).index_add_(0, inv, v)
    if kind == "split":
        a, shape = _split_input(case, seed)
        rows, cols = _grid(a, shape)
        out = []
        for r in rows:
            for c in cols:
                t = _slice(a, *r, *c)
                out.append((t[2], t[3], t[4].double()))
        return out
    a, b, rows, cols = _stage_operands(case, seed)
    rp, col, vals = _product64(a, b)
    c = (a[0], b[1], rp, col, vals)
    out = []
    for r in rows:
        for w in cols:
            out.append(_slice(c, *r, *w)[2:])
    return out


def _csr_bytes(m, nnz, ptr, width):
    return (m + 1) * ptr + nnz * (4 + width)


def work(case):
    kind = case["kind"]
    if kind == "spgemm":
        w = 8 if case["dtype"] == "f64" else 4
        a, b = _spgemm_inputs(case, 0)
        products, nnz = _product_size(a, b)
        read = _csr_bytes(a[0], a[3].numel(), case["ptr"], w)
        read += 0 if b is a else _csr_bytes(b[0], b[3].numel(), case["ptr"], w)
        return {"bytes": read + _csr_bytes(a[0], nnz, 8, w), "flops": 2 * products}
    if kind == "spmm":
        a = _matrix(case, 0, _generator(0), torch.float32)
        wc = 8 if case["b"] == "f64" else 4
        wb = {"f32": 4, "bf16": 2, "f64": 8}[case["b"]]
        nnz, n = a[3].numel(), case["cols"]
        touched = int(torch.unique(a[3]).numel())  # rows of B that A refers to
        c = a[0] * n * wc * (2 if case["beta"] else 1)
        return {"bytes": _csr_bytes(a[0], nnz, case["ptr"], wc) + touched * n * wb + c, "flops": 2 * nnz * n}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        w = 8 if case["mode"] == "f64" else 4
        return {"bytes": w * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2 * m * n * k}
    if kind == "accumulate":
        w = 8 if case["dtype"] == "f64" else 4
        tiles = _accumulate_inputs(case, 0)
        m, n = tiles[0][0], tiles[0][1]
        key = torch.cat([torch.repeat_interleave(torch.arange(m, device=DEV), t[2][1:] - t[2][:-1]) * n + t[3].long()
                         for t in tiles])
        read = sum(_csr_bytes(m, t[3].numel(), case["ptr"], w) for t in tiles)
        return {"bytes": read + _csr_bytes(m, int(torch.unique(key).numel()), 8, w), "flops": key.numel()}
    if kind == "split":
        a, shape = _split_input(case, 0)
        w = 8 if case["dtype"] == "f64" else 4
        nnz = a[3].numel()
        rows, cols = _grid(a, shape)
        out = nnz * (4 + w) + len(cols) * (a[0] + len(rows)) * 4
        return {"bytes": _csr_bytes(a[0], nnz, case["ptr"], w) + out, "flops": 0}
    a, b, rows, cols = _stage_operands(case, 0)
    products, nnz = _product_size(a, b)
    read = _csr_bytes(a[0], a[3].numel(), 4, 4) + _csr_bytes(b[0], b[3].numel(), 4, 4)
    return {"bytes": read + len(cols) * (a[0] + len(rows)) * 8 + nnz * 8, "flops": 2 * products}
