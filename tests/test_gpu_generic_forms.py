"""The generic family's forms (streaming up to 64 rows, 64x64 and 128x128 tiles above) at the edges of
their tiles, K steps and dispatch, against float64. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _codes(rows, k, pad, seed, dev):
    """[rows, k] finite e4m3fn codes of both signs at a byte offset of 1 in rows of k + pad bytes, with NaN
    codes in everything around them."""
    g = torch.Generator(device=dev).manual_seed(seed)
    table = torch.full((rows * (k + pad) + 1,), 0x7F, dtype=torch.uint8, device=dev)
    view = table[1:].view(rows, k + pad)[:, :k]
    view.copy_(torch.randn((rows, k), generator=g, device=dev).to(torch.float8_e4m3fn).view(torch.uint8))
    return view.view(torch.float8_e4m3fn)


# (m, n, k): one K byte to several 128-byte steps; rows and columns around 16, 32, 64 and 128; of the two with about
# 2050 rows the first has 510 tiles of 128x128, which is what it runs, the second 544, where 128x64 tiles are quicker
SHAPES = [(1, 1, 1), (16, 16, 15), (17, 33, 127), (32, 31, 128), (33, 40, 129), (64, 65, 4099), (65, 63, 17), (128, 129, 256),
          (129, 257, 1041), (517, 300, 383), (2049, 3840, 145), (2050, 3971, 273),
          # rows shorter than 16 bytes, in every mix of 8-, 4-, 2- and 1-byte pieces; panels on either side of the lines
          # between the streaming form and the tiles
          (3, 40, 2), (70, 33, 3), (5, 66, 5), (64, 20, 7), (16, 17, 8), (33, 70, 11), (66, 65, 13), (7, 31, 14),
          (16, 8193, 127), (17, 8193, 255), (64, 4097, 255), (64, 4096, 255), (100, 33000, 126)]


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_forms_against_float64(gpu_device, m, n, k, out_dtype):
    print(f"case m={m} n={n} k={k} {out_dtype}", flush=True)
    dev = gpu_device
    a, b = _codes(m, k, 3, 1, dev), _codes(n, k, 7, 2, dev)
    g = torch.Generator(device=dev).manual_seed(3)
    sa = torch.rand(m, generator=g, device=dev) + 0.5
    sb = torch.rand(n, generator=g, device=dev) + 0.5
    bias = torch.randn(n, generator=g, device=dev).to(torch.bfloat16)
    canvas = torch.full((m + 2, n + 5), 7.0, dtype=out_dtype, device=dev)
    out = ops.fp8_gemm_rowwise(a, b, sa, sb, bias=bias, out=canvas[1:-1, 2:-3], out_dtype=out_dtype, variant=_lib.VARIANT_GENERIC)
    torch.cuda.synchronize()
    scale = sa.double()[:, None] * sb.double()[None, :]
    exact = (a.double() @ b.double().t()) * scale + bias.double()
    # one rounding of the result (half a unit in the last place) after an f32 sum of k exact products, two
    # scalings and the bias: each adds at most 2^-24 of the magnitudes it adds up
    mant = 8 if out_dtype == torch.bfloat16 else 11
    smallest = 2.0 ** -126 if out_dtype == torch.bfloat16 else 2.0 ** -14
    half_ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=smallest))) - mant)
    slack = ((a.double().abs() @ b.double().abs().t()) * scale + bias.double().abs()) * (k + 3) * 2.0 ** -24
    excess = ((out.double() - exact).abs() - half_ulp * (1 + 2.0 ** -10) - slack).max().item()
    assert excess <= 0, f"{excess} beyond the bound"
    guard = canvas.clone()
    guard[1:-1, 2:-3] = 7.0
    assert (guard == 7.0).all()


# more columns than a launch of the streaming form holds lanes for (512 lanes for 16 columns, 2^32 lanes)
@pytest.mark.parametrize("m,n", [(1, 2**27 + 40), (1, 2**27 - 16), (3, 2**27)])
def test_columns_beyond_the_streaming_forms_grid(gpu_device, m, n):
    print(f"case m={m} n={n} k=1", flush=True)
    b = torch.arange(n, device=gpu_device, dtype=torch.int64).remainder_(13).to(torch.uint8).add_(0x38).view(torch.float8_e4m3fn).view(n, 1)
    a = torch.ones((m, 1), device=gpu_device).to(torch.float8_e4m3fn)
    sa, sb = torch.ones(m, device=gpu_device), torch.ones(n, device=gpu_device)
    got = ops.fp8_gemm_rowwise(a, b, sa, sb)
    torch.cuda.synchronize()
    assert torch.equal(got, b.to(torch.bfloat16).view(1, n).expand(m, n))
