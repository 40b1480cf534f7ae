"""The forms of the block-scaled GEMM at the edges of their tiles, K blocks and dispatch, against
float64. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops
from tritonbench_amd._lib import BLOCK_NARROW, BLOCK_ONE_TILE, BLOCK_TILES_128, BLOCK_TILES_128_STREAM, BLOCK_TILES_256

pytestmark = pytest.mark.gpu


def _expand(codes, scales):
    s = scales.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return codes.double() * s[: codes.shape[0], : codes.shape[1]]


def _run(xq, wq, xs, ws, out, form):
    """The product in `form`, whatever the library would choose for the shape (None: its choice, through the wrapper)."""
    if form is None:
        return ops.fp8_gemm_blockwise(xq, wq, xs, ws, out=out)
    m, k = xq.shape
    st = _lib.load().mi355x_fp8_blockwise_gemm_ex(
        xq.data_ptr(), wq.data_ptr(), xs.data_ptr(), ws.data_ptr(), out.data_ptr(), m, wq.shape[0], k, xq.stride(0), wq.stride(0),
        out.stride(0), form, torch.cuda.current_stream().cuda_stream)
    _lib.check(st, "mi355x_fp8_blockwise_gemm_ex")
    return out


def _streaming_forms(m, n):
    """The streaming forms that take the shape: one tile a workgroup up to 64 rows, narrow tiles where the row-wise ones go."""
    return ([BLOCK_ONE_TILE] if m <= 64 else []) + ([BLOCK_NARROW] if _lib.skinny_family_takes(m, n) else [])


def _check(m, n, k, dev, form, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    gk = -(-k // 128)
    xq = torch.randn((m, k), generator=g, device=dev).to(torch.float8_e4m3fn)
    wq = torch.randn((n, k), generator=g, device=dev).to(torch.float8_e4m3fn)
    # factors over eight binades, so that a product added with a neighbour's factor would show; one block of
    # zeros with a factor of zero
    xs = torch.exp2(torch.rand((-(-m // 128), gk), generator=g, device=dev) * 8 - 4)
    ws = torch.exp2(torch.rand((-(-n // 128), gk), generator=g, device=dev) * 8 - 4)
    if gk > 2:
        wq[:128, 128:256] = 0
        ws[0, 1] = 0.0
    canvas = torch.full((m + 2, n + 8), 7.0, dtype=torch.bfloat16, device=dev)
    aligned = n % 8 == 0
    out = canvas[1:-1, :n] if aligned else canvas[1:-1, 3 : n + 3]
    _run(xq, wq, xs, ws, out, form)
    torch.cuda.synchronize()
    a, b = _expand(xq, xs), _expand(wq, ws)
    exact = a @ b.t()
    # One rounding to bf16; f32 sums of k products with two roundings of scale per block of 128; and the fp8 matrix
    # instruction's own sum of 64 products, which aligns them to the largest before it adds: over 300k such sums it
    # was off by up to 2^-11.9 of the largest product (two instructions per block; the largest product is at most
    # the product of the rows' largest elements).
    ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=2.0**-126))) - 7)
    slack = (a.abs() @ b.abs().t()) * (k + 4 * gk + 8) * 2.0**-24
    largest = [torch.nn.functional.pad(t.abs(), (0, gk * 128 - k)).view(-1, gk, 128).amax(2) for t in (a, b)]
    slack += (largest[0] @ largest[1].t()) * 2 * 2.0**-11.5
    excess = ((out.double() - exact).abs() - ulp - slack).max().item()
    assert excess <= 0, f"{m}x{n}x{k}: {excess} beyond the bound"
    rel = ((out.double() - exact).norm() / exact.norm()).item()
    assert rel < 4e-3, f"{m}x{n}x{k}: relative error {rel} (rounding alone: 1.7e-3)"
    guard = canvas.clone()
    guard[1:-1, (slice(0, n) if aligned else slice(3, n + 3))] = 7.0
    assert (guard == 7.0).all()


# 256x256 tiles of two alternating groups of waves: one step, two, three (the depth of the ring of B), a partial last step,
# ragged rows and columns (also less than a wave's share of a tile), stores element by element, several tiles per
# workgroup and a last round that reaches few of them
@pytest.mark.parametrize("m,n,k", [(4096, 4096, 96), (4100, 4090, 144), (4350, 4100, 384), (3000, 5000, 3008), (6000, 3000, 528),
                                   (4097, 13313, 640), (8200, 4104, 1040)])
def test_large_tiles_against_float64(gpu_device, m, n, k):
    print(f"case m={m} n={n} k={k}", flush=True)
    _check(m, n, k, gpu_device, BLOCK_TILES_256)


# the streaming forms: rows around 16, 32, 48 and 64, tiles whose columns straddle two column blocks (20 and 40 columns a
# tile), column counts that are no multiple of 4, one K block, fewer K blocks than waves, partial last blocks; row
# blocks (65 .. 256 rows) in every tile size
@pytest.mark.parametrize("m,n,k", [(1, 2304, 2048), (16, 130, 96), (17, 1000, 144), (33, 515, 1040), (48, 640, 3008), (49, 300, 400),
                                   (64, 2050, 1168), (16, 5000, 8192), (30, 10007, 2000), (64, 9999, 4112), (65, 515, 1040),
                                   (128, 2300, 6656), (200, 1030, 2064), (256, 4090, 528)])
def test_streaming_forms_against_float64(gpu_device, m, n, k):
    forms = _streaming_forms(m, n)
    assert forms
    for form in forms:
        print(f"case m={m} n={n} k={k} form={form}", flush=True)
        _check(m, n, k, gpu_device, form)


# 128x128 tiles whose walk over K starts at a step of its own per tile column and wraps around (one tile row, wide panel): the
# factors' ratios have to wrap with it; one step, few steps, many steps with a partial last one
@pytest.mark.parametrize("m,n,k", [(100, 24600, 128), (128, 25000, 400), (77, 26001, 2064)])
def test_rotated_walk_against_float64(gpu_device, m, n, k):
    print(f"case m={m} n={n} k={k}", flush=True)
    _check(m, n, k, gpu_device, BLOCK_TILES_128_STREAM)


# the library's own choice for a shape well inside each form's range, and that it is what runs: the same bits as the pinned form
@pytest.mark.parametrize("m,n,k,form", [(1, 2304, 2048, BLOCK_ONE_TILE), (32, 8192, 8192, BLOCK_NARROW), (128, 8192, 8192, BLOCK_NARROW),
                                        (64, 57344, 8192, BLOCK_TILES_128_STREAM), (512, 1024, 1024, BLOCK_TILES_128),
                                        (4096, 4096, 4096, BLOCK_TILES_256)])
def test_the_choice_runs_the_form_it_names(gpu_device, m, n, k, form):
    assert _lib.load().mi355x_fp8_blockwise_form(m, n, k) == form
    g = torch.Generator(device=gpu_device).manual_seed(7)
    code = lambda r: torch.randn((r, k), generator=g, device=gpu_device).to(torch.float8_e4m3fn)
    factors = lambda r: torch.rand((-(-r // 128), -(-k // 128)), generator=g, device=gpu_device) + 0.5
    x, w, xs, ws = code(m), code(n), factors(m), factors(n)
    out = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
    assert torch.equal(_run(x, w, xs, ws, None, None), _run(x, w, xs, ws, out, form))


@pytest.mark.parametrize("m,n,form", [(65, 512, BLOCK_ONE_TILE), (257, 512, BLOCK_NARROW), (128, 20000, BLOCK_NARROW)])
def test_a_form_refuses_what_it_does_not_take(gpu_device, m, n, form):
    x, w = (torch.ones((r, 256), device=gpu_device).to(torch.float8_e4m3fn) for r in (m, n))
    xs, ws = (torch.ones((-(-r // 128), 2), device=gpu_device) for r in (m, n))
    with pytest.raises(NotImplementedError):
        _run(x, w, xs, ws, torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device), form)


# An infinite factor (what the block quantiser returns for a block that holds an infinity) in the last K block, against products that
# are not zero: the result is that infinity in every form, also where a step of K reaches past the last block.
@pytest.mark.parametrize("side", ["a", "b"])
@pytest.mark.parametrize("m,n,k", [(16, 130, 96), (33, 515, 1040), (48, 640, 3008), (64, 9999, 4112), (30, 10007, 2000), (16, 5000, 8192),
                                   (128, 2300, 6656), (200, 1030, 2064), (256, 4090, 528), (77, 26001, 2064), (300, 700, 528),
                                   (4096, 4096, 96), (4350, 4100, 384)])
def test_an_infinite_factor_of_the_last_block(gpu_device, m, n, k, side):
    print(f"case m={m} n={n} k={k} {side}", flush=True)
    one = torch.ones(1, device=gpu_device).to(torch.float8_e4m3fn)
    xq, wq = one.expand(m * k).clone().view(m, k), one.expand(n * k).clone().view(n, k)
    xs = torch.ones((-(-m // 128), -(-k // 128)), device=gpu_device)
    ws = torch.ones((-(-n // 128), -(-k // 128)), device=gpu_device)
    (xs if side == "a" else ws)[0, -1] = float("inf")
    want = torch.full((m, n), float(k), dtype=torch.float64, device=gpu_device)
    want[(slice(0, 128), slice(None)) if side == "a" else (slice(None), slice(0, 128))] = float("inf")
    want = want.to(torch.bfloat16)
    for form in [None, BLOCK_TILES_128, BLOCK_TILES_128_STREAM, BLOCK_TILES_256, *_streaming_forms(m, n)]:
        got = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
        assert torch.equal(_run(xq, wq, xs, ws, got, form), want), form
