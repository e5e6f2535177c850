"""What kvmix_linear_rows_supported answers (no GPU needed)."""
import pytest

from kvmix_amd import _lib, ops


@pytest.mark.parametrize("epilogue", [_lib.LINEAR_PLAIN, _lib.LINEAR_FLOAT, _lib.LINEAR_RESIDUAL, _lib.LINEAR_SWIGLU])
@pytest.mark.parametrize("m", [0, 1, 16])
def test_no_rows_of_weights(epilogue, m):
    assert ops.linear_rows_supported(m, 4096, 0, epilogue) == ops.linear_rows_supported(m, 4096, 8, epilogue)
