"""Row offsets at the edges of the one-workgroup scan (64 counts per instruction, 1024 per wavefront, 16384 per step, 32768
in all): A times the identity must return A, with rows of 0 to 2 entries and one long row at the end."""
import numpy as np
import pytest

from bcl_amd.csr import CSR
from bcl_amd.device import DeviceCSR, spgemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 63, 65, 255, 1023, 1025, 16383, 16385, 32511, 32767, 32769])
def test_offsets(handle, m):
    n = 512
    rng = np.random.default_rng(m)
    lens = np.arange(m) % 3
    lens[-1] = 300
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    col = np.concatenate([np.sort(rng.choice(n, int(x), replace=False)) for x in lens]).astype(np.int32)
    a = CSR(m, n, rp, col, rng.uniform(1, 2, col.size).astype(np.float32))
    eye = CSR(n, n, np.arange(n + 1, dtype=np.int64), np.arange(n, dtype=np.int32), np.ones(n, np.float32))
    c = spgemm(handle, DeviceCSR.from_host(a), DeviceCSR.from_host(eye)).to_host()
    np.testing.assert_array_equal(c.row_ptr, a.row_ptr)
    np.testing.assert_array_equal(c.col_idx, a.col_idx)
    np.testing.assert_array_equal(c.vals, a.vals)
