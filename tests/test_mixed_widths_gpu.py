"""A batch of products of unlike widths: one tile wider than 2^19 columns gives the whole batch's heavy rows to the
wide-tile kernel (a dense accumulator in HBM), so rows of narrow tiles that fit an LDS hash table stay there, however many
products they have. A batch of narrow tiles gives them to the rank-slice kernel. Results equal the oracle's either way."""
import numpy as np
import pytest
import torch

import oracle_py as O
from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR
from bcl_amd.stage import BATCHED_EXACT, LEARNED, StagePlan
from conftest import spgemm_value_bound

pytestmark = pytest.mark.gpu


def _csr(rows, n, rng):
    rp = np.concatenate([[0], np.cumsum([len(x) for x in rows])]).astype(np.int64)
    col = np.concatenate([np.asarray(x, np.int64) for x in rows]).astype(np.int32)
    return CSR(len(rows), n, rp, col, rng.uniform(-1, 1, col.size).astype(np.float32))


@pytest.mark.parametrize("mode", [BATCHED_EXACT, LEARNED])
@pytest.mark.parametrize("wide", [False, True])
def test_hash_rows_of_narrow_tiles(handle, mode, wide):
    rng = np.random.default_rng(4)
    k, narrow = 400, 3000  # rows of 12800 products and 2900 to 3000 entries
    brows = [np.sort(rng.choice(narrow, 128, replace=False)) for _ in range(k)]
    arows = [np.sort(rng.choice(k, 100, replace=False)) for _ in range(70)]
    other = [np.sort(rng.choice((1 << 19) + 5 if wide else 1 << 19, 20, replace=False)) for _ in range(k)]
    pairs = [(_csr(arows, k, rng), _csr(brows, narrow, rng)),
             (_csr([np.sort(rng.choice(k, 2, replace=False)) for _ in range(300)], k, rng),
              _csr(other, (1 << 19) + 5 if wide else 1 << 19, rng))]
    print(f"[mixed] mode {mode} wide {wide}", flush=True)
    plan = StagePlan(handle, [DeviceCSR.from_host(a) for a, _ in pairs], [DeviceCSR.from_host(b) for _, b in pairs],
                     mode=mode)
    plan.execute()
    torch.cuda.synchronize()
    heavy = plan.stats()["heavy_rows"]
    for p, (a, b) in enumerate(pairs):
        c, ref, c64 = plan.result_host(p), O.spgemm(a, b), O.spgemm_f64(a, b)
        np.testing.assert_array_equal(c.row_ptr, ref.row_ptr)
        np.testing.assert_array_equal(c.col_idx, ref.col_idx)
        pos = [CSR(x.m, x.n, x.row_ptr, x.col_idx, np.abs(x.vals)) for x in (a, b)]
        bound = spgemm_value_bound(a, b, c64.vals, O.spgemm_f64(*pos).vals, np.float32)
        assert (np.abs(c.vals.astype(np.float64) - c64.vals) <= bound).all()
    plan.close()
    print("[mixed] heavy rows", heavy, flush=True)
    assert (heavy == 0) == wide
