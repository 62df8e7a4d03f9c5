"""SpMM at widths whose rows of B are not whole cache lines, around the limits of their slices (64 and 128 columns) and where
the last slice is half used; the cases and the exact comparison are those of the row tests."""
import pytest

from test_spmm_rows_gpu import test_rows as compare_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,b_dtype,n,ptr", [
    ("mixed", "f64", 33, 4), ("mixed", "f64", 65, 4), ("mixed", "f64", 100, 8), ("many", "f64", 127, 4), ("mixed", "f64", 129, 4),
    ("mixed", "f64", 192 + 1, 4), ("mixed", "f64", 255, 8), ("one row", "f64", 67, 4), ("short", "f64", 66, 8),
    ("many", "f32", 33, 4), ("mixed", "f32", 63, 8), ("many", "f32", 129, 4), ("one row", "f32", 100, 4),
])
def test_unaligned_widths(handle, name, b_dtype, n, ptr):
    compare_rows(handle, name, b_dtype, n, ptr)
