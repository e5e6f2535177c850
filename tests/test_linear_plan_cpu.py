"""What kvmix_linear_rows_supported answers (no GPU needed)."""
import pytest

from kvmix_amd import _lib, ops


@pytest.mark.parametrize("epilogue", [_lib.LINEAR_PLAIN, _lib.LINEAR_FLOAT, _lib.LINEAR_RESIDUAL, _lib.LINEAR_SWIGLU])
@pytest.mark.parametrize("m", [0, 1, 16])
def test_no_rows_of_weights(epilogue, m):
    assert ops.linear_rows_supported(m, 4096, 0, epilogue) == ops.linear_rows_supported(m, 4096, 8, epilogue)


def instances():
    """The (chunks of 128 per wave, groups of four sequences, norm, epilogue) that csrc/linear_rows.hip holds a kernel for."""
    for ch, mg in ((2, 1), (2, 2), (2, 4), (4, 1), (4, 2), (4, 4), (6, 1), (6, 2), (6, 4), (8, 1), (8, 2), (11, 1), (11, 2), (14, 1)):
        for epi in (_lib.LINEAR_PLAIN, _lib.LINEAR_FLOAT, _lib.LINEAR_RESIDUAL):
            yield ch, mg, False, epi
        for epi in (_lib.LINEAR_PLAIN, _lib.LINEAR_FLOAT):
            if ch <= 8 and (ch <= 4 or mg <= 2):
                yield ch, mg, True, epi
        for epi in (_lib.LINEAR_SWIGLU, _lib.LINEAR_ROPE_APPEND):
            if ch <= 8 and (ch <= 4 or mg <= 2):
                yield ch, mg, False, epi
            if ch <= 8 and (ch <= 4 or mg == 1 or (ch <= 6 and mg <= 2)):
                yield ch, mg, True, epi


@pytest.mark.parametrize("epilogue", range(5))
@pytest.mark.parametrize("norm", [False, True])
def test_query_says_yes_only_where_there_is_a_kernel(epilogue, norm):
    have = set(instances())
    for ch in (2, 4, 6, 8, 11, 14):
        for mg in (1, 2, 4):
            yes = ops.linear_rows_supported(4 * mg, 1024 * ch, 256, epilogue, norm, 128, 256)
            assert not yes or (ch, mg, norm, epilogue) in have, (ch, mg)
            if ch <= 4:
                assert yes == ((ch, mg, norm, epilogue) in have)
