"""The block-scaled entries' host arithmetic: which forms they refuse, and that a form named before any device call. No device needed."""
import ctypes

import pytest

from tritonbench_amd import _lib


def _status(entry, form, *space):
    codes, factors, out = (ctypes.create_string_buffer(128 * 1024 + 64) for _ in range(3))
    at = lambda b: -(-ctypes.addressof(b) // 64) * 64
    return entry(at(codes), at(codes), at(factors), at(factors), at(out), 64, 64, 1024, 1024, 1024, 64, *space, form, None)


# the entry without a workspace knows the five forms; a factor (form + 256 * s) is the other entry's
@pytest.mark.parametrize("form", [5, 255, 256, _lib.BLOCK_TILES_128 + 256, _lib.BLOCK_TILES_128 + 256 * 2, _lib.BLOCK_NARROW + 256, 1 << 30])
def test_the_entry_without_a_workspace_refuses_factors(form):
    assert _status(_lib.load().mi355x_fp8_blockwise_gemm_ex, form) == _lib.EINVAL


@pytest.mark.parametrize("form", [5, 255, _lib.BLOCK_TILES_256 + 256 * 2, _lib.BLOCK_TILES_128 + 256 * 2])
def test_the_entry_with_a_workspace_refuses_other_forms_and_factors_without_space(form):
    assert _status(_lib.load().mi355x_fp8_blockwise_gemm_ws, form, None, 0) == _lib.EINVAL
