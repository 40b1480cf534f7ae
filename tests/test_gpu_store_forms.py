"""How the tiles store C (streaming on the 128-byte lines, ordinary aligned, pieces that start at any 2 bytes): the kind
changes where the bytes of a row lie and no value, so every placement of C has to hold the bits of one on the lines, and
nothing beside them. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu

# column offset and pitch beyond N of C in a wider canvas, in elements of 2 bytes: any 2, 4, 8 bytes; 16 bytes off the lines
PLACES = [(1, 6), (2, 12), (4, 8), (8, 24), (3, 5)]


def _codes(rows, k, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn((rows, k), generator=g, device=dev).to(torch.float8_e4m3fn)


def _place(m, n, offset, extra, dtype, dev):
    """C inside a canvas of sevens, `offset` elements into rows of n + extra (and a row above and below)."""
    canvas = torch.full(((m + 2) * (n + extra) + 64,), 7.0, dtype=dtype, device=dev)
    rows = canvas[: (m + 2) * (n + extra)].view(m + 2, n + extra)
    return canvas, rows[1:-1, offset : offset + n]


def _on_lines(m, n, dtype, dev):
    return torch.empty((m, -(-n // 64) * 64), dtype=dtype, device=dev)[:, :n]


def _check(run, m, n, dtype, dev, places):
    want = run(_on_lines(m, n, dtype, dev)).clone()
    for offset, extra in places:
        print(f"case {m}x{n} offset {offset} pitch {n + extra}", flush=True)
        canvas, c = _place(m, n, offset, extra, dtype, dev)
        run(c)
        torch.cuda.synchronize()
        assert torch.equal(c.view(torch.int16), want.view(torch.int16)), (offset, extra)
        c.fill_(7.0)
        assert (canvas == 7.0).all(), (offset, extra)


# columns that leave 0 to 7 of a lane's eight, rows around the tiles' edges, by tile configuration
@pytest.mark.parametrize("config", range(7))
@pytest.mark.parametrize("m,n", [(257, 261), (129, 386), (65, 255), (300, 264)])
def test_tiles_at_any_place(gpu_device, config, m, n):
    dev, k = gpu_device, 272
    a, b = _codes(m, k, 1, dev), _codes(n, k, 2, dev)
    sa, sb = torch.rand(m, device=dev) + 0.5, torch.rand(n, device=dev) + 0.5
    bias = torch.randn(n, device=dev).to(torch.bfloat16)
    variant = _lib.VARIANT_TILED | ((config + 1) << 8) | (1 << 16)
    for dtype, add in ((torch.bfloat16, bias), (torch.float16, None)):
        _check(lambda c: ops.fp8_gemm_rowwise(a, b, sa, sb, bias=add, out=c, variant=variant, out_dtype=dtype), m, n, dtype, dev, PLACES)


@pytest.mark.parametrize("n", [257, 386, 519])
def test_grouped_tiles_at_any_place(gpu_device, n):
    dev, m, k = gpu_device, 700, 272
    a, b = _codes(m, k, 1, dev), _codes(3 * n, k, 2, dev)
    sa, sb = torch.rand(m, device=dev) + 0.5, torch.rand(3 * n, device=dev) + 0.5
    sizes = torch.tensor([301, 0, 399], dtype=torch.int32, device=dev)
    for config in range(3):
        _check(lambda c: ops.fp8_gemm_rowwise_grouped(a, b, sizes, sa, sb, out=c, tile_config=config), m, n, torch.bfloat16, dev, PLACES)


@pytest.mark.parametrize("form", [_lib.BLOCK_TILES_128, _lib.BLOCK_TILES_256])
@pytest.mark.parametrize("m,n", [(257, 261), (130, 386)])
def test_block_scaled_tiles_at_any_place(gpu_device, form, m, n):
    dev, k = gpu_device, 272
    a, b = _codes(m, k, 1, dev), _codes(n, k, 2, dev)
    xs, ws = torch.rand((-(-m // 128), 3), device=dev) + 0.5, torch.rand((-(-n // 128), 3), device=dev) + 0.5

    def run(c):
        st = _lib.load().mi355x_fp8_blockwise_gemm_ex(a.data_ptr(), b.data_ptr(), xs.data_ptr(), ws.data_ptr(), c.data_ptr(), m, n, k,
                                                      k, k, c.stride(0), form, torch.cuda.current_stream().cuda_stream)
        _lib.check(st, "mi355x_fp8_blockwise_gemm_ex")
        return c

    _check(run, m, n, torch.bfloat16, dev, PLACES)


# a C of more than 48 MB, on and off the lines: ordinary stores
@pytest.mark.parametrize("m,n", [(3070, 8328), (6150, 4136)])
def test_large_result_off_the_lines(gpu_device, m, n):
    dev, k = gpu_device, 144
    a, b = _codes(m, k, 1, dev), _codes(n, k, 2, dev)
    sa, sb = torch.rand(m, device=dev) + 0.5, torch.rand(n, device=dev) + 0.5
    for dtype in (torch.bfloat16, torch.float16):
        _check(lambda c: ops.fp8_gemm_rowwise(a, b, sa, sb, out=c, out_dtype=dtype, variant=_lib.VARIANT_TILED), m, n, dtype, dev, [(8, 24), (0, 0)])
    xs, ws = torch.rand((-(-m // 128), 2), device=dev) + 0.5, torch.rand((-(-n // 128), 2), device=dev) + 0.5
    _check(lambda c: ops.fp8_gemm_blockwise(a, b, xs, ws, out=c), m, n, torch.bfloat16, dev, [(8, 24), (0, 0)])


# split K with rows of partial sums that start on any 4 bytes: the columns of a panel that ends on 4 of them hold the same bits
@pytest.mark.parametrize("config", range(7))
@pytest.mark.parametrize("m,n,splits", [(3, 1, 2), (65, 129, 3), (130, 254, 2), (257, 515, 5), (300, 3, 4)])
def test_partial_rows_off_sixteen_bytes(gpu_device, config, m, n, splits):
    print(f"case {m}x{n} config {config} splits {splits}", flush=True)
    dev, k = gpu_device, 1168
    wide = -(-n // 4) * 4
    a, b = _codes(m, k, 1, dev), _codes(wide, k, 2, dev)
    sa, sb = torch.rand(m, device=dev) + 0.5, torch.rand(wide, device=dev) + 0.5
    bias = torch.randn(wide, device=dev).to(torch.bfloat16)
    variant = _lib.VARIANT_TILED | ((config + 1) << 8) | (splits << 16)
    want = ops.fp8_gemm_rowwise(a, b, sa, sb, bias=bias, variant=variant)[:, :n]
    space = torch.full((splits * m * n + 256,), 7.0, device=dev)
    canvas, c = _place(m, n, 1, 6, torch.bfloat16, dev)
    ops.fp8_gemm_rowwise(a, b[:n], sa, sb[:n], bias=bias[:n], out=c, variant=variant, workspace=space[: splits * m * n].view(torch.uint8))
    torch.cuda.synchronize()
    assert torch.equal(c.view(torch.int16), want.view(torch.int16))
    c.fill_(7.0)
    assert (canvas == 7.0).all() and (space[splits * m * n :] == 7.0).all()


# (four rows a thread in the second pass: more than 2048 workgroups of 256 lanes with one)
def test_second_pass_with_four_rows_off_sixteen_bytes(gpu_device):
    dev, m, n, k = gpu_device, 1027, 2054, 272
    a, b = _codes(m, k, 1, dev), _codes(n + 2, k, 2, dev)
    sa, sb = torch.rand(m, device=dev) + 0.5, torch.rand(n + 2, device=dev) + 0.5
    variant = _lib.tiled_variant(1, 2)
    want = ops.fp8_gemm_rowwise(a, b, sa, sb, variant=variant)[:, :n]
    got = ops.fp8_gemm_rowwise(a, b[:n], sa, sb[:n], variant=variant)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16).contiguous())
