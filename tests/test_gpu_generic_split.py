"""The generic family with K cut into parts, and its 128x64 tiles, at the edges of tiles and parts, against float64.
Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _operands(m, n, k, dev):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, b = (torch.randn((r, k), generator=g, device=dev).to(torch.float8_e4m3fn) for r in (m, n))
    sa, sb = (torch.rand(r, generator=g, device=dev) + 0.5 for r in (m, n))
    bias = torch.randn(n, generator=g, device=dev).to(torch.bfloat16)
    scale = sa.double()[:, None] * sb.double()[None, :]
    exact = (a.double() @ b.double().t()) * scale + bias.double()
    magnitude = (a.double().abs() @ b.double().abs().t()) * scale + bias.double().abs()
    return a, b, sa, sb, bias, exact, magnitude


def _check(out, exact, magnitude, k):
    # one rounding of the result (half a unit in the last place) after an f32 sum of k exact products in any order, two
    # scalings and the bias: each adds at most 2^-24 of the magnitudes it adds up
    half_ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=2.0 ** -14))) - 11)
    excess = ((out.double() - exact).abs() - half_ulp * (1 + 2.0 ** -10) - magnitude * (k + 3) * 2.0 ** -24).max().item()
    assert excess <= 0, f"{excess} beyond the bound"


# rows and columns around 64 and 128, fewer than four columns, rows of partial sums that start on any 4 bytes; a last part that is
# the partial step alone (49 steps in thirteen parts), one without it (K a multiple of 128), one that is shorter than the others
@pytest.mark.parametrize("m,n,k", [(65, 3, 9001), (129, 65, 4097), (70, 701, 5003), (100, 64, 33 * 128), (200, 300, 6145),
                                   (128, 130, 48 * 128 + 1), (66, 1, 3333), (257, 190, 8200), (246, 1568, 6290)])
@pytest.mark.parametrize("space", ["whole", "two planes", "none", "misaligned"])
def test_parts_against_float64(gpu_device, m, n, k, space):
    print(f"case m={m} n={n} k={k} {space}", flush=True)
    need = _lib.load().mi355x_fp8_rowwise_workspace_bytes(m, n, k, _lib.VARIANT_GENERIC)
    assert need >= 2 * m * n * 4 and need % (m * n * 4) == 0
    a, b, sa, sb, bias, exact, magnitude = _operands(m, n, k, gpu_device)
    size = {"whole": need, "two planes": 2 * m * n * 4 + 5, "none": 1, "misaligned": need + 4}[space]
    # (guards around the workspace that was promised, NaN in it)
    canvas = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device=gpu_device)
    at = 2048 + (4 if space == "misaligned" else 0)
    out = ops.fp8_gemm_rowwise(a, b, sa, sb, bias=bias, out_dtype=torch.float16, variant=_lib.VARIANT_GENERIC,
                               workspace=canvas[at:2048 + size])
    torch.cuda.synchronize()
    _check(out, exact, magnitude, k)
    assert (canvas[:2048] == 0xFF).all() and (canvas[2048 + size:] == 0xFF).all()
    if space in ("none", "misaligned"):
        assert (canvas == 0xFF).all()


# each form of the tiles with ragged edges, 255 64x64 tiles and 272
@pytest.mark.parametrize("m,n,k,form", [(129, 64 * 160 - 1, 131, _lib.GENERIC_TILES_64), (129, 64 * 159, 257, _lib.GENERIC_TILES_64),
                                        (2049, 64 * 20 + 1, 700, _lib.GENERIC_TILES_64), (1025, 7200, 2065, _lib.GENERIC_TILES_64),
                                        (1025, 897, 1041, _lib.GENERIC_TILES_64_K), (1025, 961, 1041, _lib.GENERIC_TILES_128X64_K),
                                        (2049, 1857, 1041, _lib.GENERIC_TILES_128_K), (2049, 3713, 1041, _lib.GENERIC_TILES_128)])
def test_tile_forms_against_float64(gpu_device, m, n, k, form):
    print(f"case m={m} n={n} k={k}", flush=True)
    assert _lib.load().mi355x_fp8_rowwise_generic_form(m, n, k, k % 4 == 0) == form
    a, b, sa, sb, bias, exact, magnitude = _operands(m, n, k, gpu_device)
    _check(ops.fp8_gemm_rowwise(a, b, sa, sb, bias=bias, out_dtype=torch.float16, variant=_lib.VARIANT_GENERIC), exact, magnitude, k)
