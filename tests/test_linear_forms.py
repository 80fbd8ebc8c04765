"""Which products take the int8 digits (crucible_linear_workspace_bytes, 0 where they do not): shapes
on both sides of the lines of the cost rule, the measured us of the forms beside them, and the
bounds of the form itself."""
import pytest

from crucible_amd import _lib


@pytest.mark.parametrize("rows,n_out,k_in,norm,swiglu,digits", [
    (1003, 2048, 768, 1, 1, True),      # 61 against 125 (f64 tiles)
    (200, 768, 768, 0, 0, False),       # 23.5 against 13.8 (decode tilings)
    (48, 50304, 768, 1, 0, True),       # 82 against 107 (tilings), 123 (f64 tiles)
    (64, 4096, 4096, 0, 0, False),      # 81 against 62 (tilings)
    (127, 4096, 4096, 0, 0, True),      # 81 against 115 (tilings)
    (64, 11008, 4096, 1, 1, True),      # 207 against 308 (f64 tiles)
    (8000, 4096, 64, 0, 0, False),      # 114 against 100 (f64 tiles)
    (8000, 64, 4096, 0, 0, False),      # 171 against 115 (tilings)
    (8000, 256, 256, 0, 0, False),      # 30 against 25 (f64 tiles)
    (32, 50304, 768, 1, 0, False),      # a decode batch
    (4000, 768, 96, 0, 0, False),       # K not a multiple of 64
    (4000, 768, 16448, 0, 0, False),    # past the int32 sums
    (0, 768, 768, 0, 0, False),
])
def test_products_on_digits(rows, n_out, k_in, norm, swiglu, digits):
    lib = _lib.load()
    assert (lib.crucible_linear_workspace_bytes(rows, n_out, k_in, norm, swiglu) > 0) == digits
