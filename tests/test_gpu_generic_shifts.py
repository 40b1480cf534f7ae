"""Tiles of the generic family on rows that start at each byte of a dword: the bytes are fetched in whole dwords and, where not all rows start on
one, moved into place, so what lies in front of, between and behind the rows must not show. Each form of the tiles, K at both ends of a 128-byte step."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu

# 64x64, 128x64 and 128x128 tiles whose waves share out K, then 128x128 and 64x64 tiles whose waves share out the tile
FORMS = {
    _lib.GENERIC_TILES_64_K: [(130, 190, 640), (130, 190, 641), (130, 190, 767)],
    _lib.GENERIC_TILES_128X64_K: [(517, 3001, 896), (517, 3001, 897), (517, 3001, 1023)],
    _lib.GENERIC_TILES_128_K: [(900, 2990, 3968), (900, 2990, 3969), (900, 2990, 4095)],
    _lib.GENERIC_TILES_128: [(1100, 20011, 256), (1100, 20011, 257), (1100, 20011, 383)],
    _lib.GENERIC_TILES_64: [(130, 3000, 128), (130, 3000, 129), (130, 3000, 255), (130, 3000, 256)],
}


# where all rows start on a dword: 64x64, 128x64 and 128x128 tiles whose waves share out K, then 128x128, 64x64 and 128x64 whose waves share out the tile
FORMS_ON_DWORDS = {
    **{f: FORMS[f] for f in (_lib.GENERIC_TILES_64_K, _lib.GENERIC_TILES_128X64_K, _lib.GENERIC_TILES_128, _lib.GENERIC_TILES_64)},
    _lib.GENERIC_TILES_128_K: [(193, 13249, 640), (193, 13249, 641), (193, 13249, 767)],
    _lib.GENERIC_TILES_128X64: [(745, 5384, 640), (745, 5384, 641), (745, 5384, 767)],
}


@pytest.mark.parametrize("m,n,k,form", [(*s, form) for form, shapes in FORMS.items() for s in shapes])
@pytest.mark.parametrize("shift,pitch", [(1, 0), (2, 3), (3, 2), (0, 1)])
def test_rows_at_any_byte(gpu_device, m, n, k, form, shift, pitch):
    if shift or (k + pitch) % 4:
        assert _lib.load().mi355x_fp8_rowwise_generic_form(m, n, k, 0) == form
    _check(gpu_device, m, n, k, shift, pitch)


@pytest.mark.parametrize("m,n,k,form", [(*s, form) for form, shapes in FORMS_ON_DWORDS.items() for s in shapes])
@pytest.mark.parametrize("shift,pad", [(0, 0), (4, 4), (8, 20)])
def test_rows_on_dwords(gpu_device, m, n, k, form, shift, pad):
    assert _lib.load().mi355x_fp8_rowwise_generic_form(m, n, k, 1) == form
    _check(gpu_device, m, n, k, shift, -k % 4 + pad)


def _check(gpu_device, m, n, k, shift, pitch):
    assert _lib.load().mi355x_fp8_rowwise_workspace_bytes(m, n, k, _lib.VARIANT_GENERIC) == 0  # (in one piece)
    print(f"case m={m} n={n} k={k} shift={shift} pitch={pitch}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(m + n + k)

    def operand(rows):
        """Codes between NaN codes, from byte `shift` on."""
        ld = k + pitch
        codes = torch.randn((rows, k), generator=g, device=gpu_device).to(torch.float8_e4m3fn)
        canvas = torch.full((rows * ld + 64,), 0x7F, dtype=torch.uint8, device=gpu_device)
        view = canvas[16 + shift : 16 + shift + rows * ld].view(rows, ld)[:, :k]
        view.copy_(codes.view(torch.uint8))
        return view.view(torch.float8_e4m3fn), codes.float()

    (a, fa), (b, fb) = operand(m), operand(n)
    sa, sb = (torch.rand(r, generator=g, device=gpu_device) + 0.5 for r in (m, n))
    out = ops.fp8_gemm_rowwise(a, b, sa, sb, out_dtype=torch.float16, variant=_lib.VARIANT_GENERIC).double()
    fa, fb = fa.double() * sa.double()[:, None], fb.double() * sb.double()[:, None]
    exact = fa @ fb.t()
    # one rounding to binary16 (2^-11 of the value) and f32 sums of K products, off by at most K * 2^-24 of the sum of magnitudes
    assert ((out - exact).abs() <= 2.0**-11 * exact.abs() + 2 * k * 2.0**-24 * (fa.abs() @ fb.abs().t()) + 1e-6).all()
