"""The block-scaled entries' host arithmetic: which forms they refuse, and that a form named before any device call. No device needed."""
import ctypes

import pytest

from tritonbench_amd import _lib


def _status(entry, form, *space, shape=(64, 64, 1024)):
    codes, factors, out = (ctypes.create_string_buffer(128 * 1024 + 64) for _ in range(3))
    at = lambda b: -(-ctypes.addressof(b) // 64) * 64
    m, n, k = shape
    return entry(at(codes), at(codes), at(factors), at(factors), at(out), m, n, k, k, k, n, *space, form, None)


# the entry without a workspace knows its forms by name; a factor (form + 256 * s) is the other entry's
@pytest.mark.parametrize("form", [5, 255, 256, _lib.BLOCK_TILES_128 + 256, _lib.BLOCK_TILES_128 + 256 * 2, _lib.BLOCK_NARROW + 256, 1 << 30])
def test_the_entry_without_a_workspace_refuses_factors(form):
    assert _status(_lib.load().mi355x_fp8_blockwise_gemm_ex, form) == _lib.EINVAL


@pytest.mark.parametrize("form", [5, 255, _lib.BLOCK_TILES_256 + 256 * 2, _lib.BLOCK_TILES_128 + 256 * 2])
def test_the_entry_with_a_workspace_refuses_other_forms_and_factors_without_space(form):
    assert _status(_lib.load().mi355x_fp8_blockwise_gemm_ws, form, None, 0) == _lib.EINVAL


# what the query names can be pinned, and is what the library's choice runs: the form that keeps A on chip has a name of its own
@pytest.mark.parametrize("m,n,k", [(16, 8192, 8192), (16, 144, 8192), (9, 160, 6160), (16, 4240, 2000), (16, 8192, 3600), (11, 8000, 6000)])
def test_the_form_that_keeps_a_on_chip_is_named(m, n, k):
    assert _lib.load().mi355x_fp8_blockwise_form(m, n, k) == _lib.BLOCK_RESIDENT


# (where it is 7 to 15 % behind one tile a workgroup)
@pytest.mark.parametrize("m,n,k", [(2, 1600, 3648), (16, 2528, 3264), (4, 336, 3376), (8, 1088, 4592), (4, 5376, 3584), (2, 256, 3600), (8, 320, 3536)])
def test_the_form_that_keeps_a_on_chip_is_left_where_it_is_behind(m, n, k):
    assert _lib.load().mi355x_fp8_blockwise_form(m, n, k) == _lib.BLOCK_ONE_TILE


@pytest.mark.parametrize("shape", [(17, 64, 1024), (16, 72, 1024), (16, 8208, 64), (16, 16, 8208)])
def test_the_form_that_keeps_a_on_chip_refuses_what_it_does_not_take(shape):
    assert _status(_lib.load().mi355x_fp8_blockwise_gemm_ex, _lib.BLOCK_RESIDENT, shape=shape) == _lib.ENOTSUP
