"""The block-scaled GEMM with K cut into parts: pinned factors at the edges of tiles, K blocks and parts against float64, and the
plans of the library itself. Needs an MI355X."""
import pytest
import torch

from test_gpu_blockwise_forms import _expand
from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _call(xq, wq, xs, ws, out, space, form):
    lib = _lib.load()
    return lib.mi355x_fp8_blockwise_gemm_ws(
        xq.data_ptr(), wq.data_ptr(), xs.data_ptr(), ws.data_ptr(), out.data_ptr(), xq.shape[0], wq.shape[0], xq.shape[1], xq.stride(0),
        wq.stride(0), out.stride(0), space.data_ptr() if space is not None else None, space.numel() * 4 if space is not None else 0, form,
        torch.cuda.current_stream().cuda_stream)


def _inputs(m, n, k, dev, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    gk = -(-k // 128)
    xq = torch.randn((m, k), generator=g, device=dev).to(torch.float8_e4m3fn)
    wq = torch.randn((n, k), generator=g, device=dev).to(torch.float8_e4m3fn)
    # factors over eight binades: a part that starts or ends in another part's units would show; a block of zeros with a factor of zero
    xs = torch.exp2(torch.rand((-(-m // 128), gk), generator=g, device=dev) * 8 - 4)
    ws = torch.exp2(torch.rand((-(-n // 128), gk), generator=g, device=dev) * 8 - 4)
    if gk > 2:
        wq[:128, 128:256] = 0
        ws[0, 1] = 0.0
    return xq, wq, xs, ws


def _within_bounds(out, xq, wq, xs, ws, parts):
    k = xq.shape[1]
    gk = -(-k // 128)
    a, b = _expand(xq, xs), _expand(wq, ws)
    exact = a @ b.t()
    # one rounding to bf16; f32 sums of k products with two roundings of scale per block, and of the parts; the fp8 matrix
    # instruction's own alignment of 64 products to the largest (2^-11.9 of it measured, two instructions a block)
    ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=2.0**-126))) - 7)
    slack = (a.abs() @ b.abs().t()) * (k + 4 * gk + 2 * parts + 8) * 2.0**-24
    largest = [torch.nn.functional.pad(t.abs(), (0, gk * 128 - k)).view(-1, gk, 128).amax(2) for t in (a, b)]
    slack += (largest[0] @ largest[1].t()) * 2 * 2.0**-11.5
    assert ((out.double() - exact).abs() - ulp - slack).max().item() <= 0
    assert ((out.double() - exact).norm() / exact.norm()).item() < 4e-3


# parts of one step, of an uneven last one, with a partial last step; 16 steps a part and more take the deeper ring; more
# than 256 items two workgroups a CU
@pytest.mark.parametrize("m,n,k,splits", [(1, 1, 144, 2), (128, 128, 256, 2), (129, 130, 1040, 3), (300, 520, 1168, 9), (65, 255, 2048, 16),
                                          (257, 387, 4624, 2), (130, 640, 4096, 2), (1100, 1000, 1536, 5), (40, 129, 32768, 16)])
def test_pinned_factor_against_float64(gpu_device, m, n, k, splits):
    print(f"case {m}x{n}x{k} in {splits}", flush=True)
    xq, wq, xs, ws = _inputs(m, n, k, gpu_device)
    canvas = torch.full((m + 2, n + 5), 7.0, dtype=torch.bfloat16, device=gpu_device)
    space = torch.full((splits * m * n + 64,), 7.0, device=gpu_device)
    out = canvas[1:-1, 2:-3]
    _lib.check(_call(xq, wq, xs, ws, out, space[:-64], _lib.BLOCK_TILES_128 + 256 * splits), "gemm_ws")
    torch.cuda.synchronize()
    _within_bounds(out, xq, wq, xs, ws, splits)
    out.fill_(7.0)
    assert (canvas == 7.0).all() and (space[-64:] == 7.0).all()


@pytest.mark.parametrize("m,n,k", [(312, 512, 9088), (59, 655, 26112)])
def test_the_wrapper_cuts_k_and_may_be_captured(gpu_device, m, n, k):
    xq, wq, xs, ws = _inputs(m, n, k, gpu_device)
    need = _lib.load().mi355x_fp8_blockwise_workspace_bytes(m, n, k)
    assert need >= 2 * 4 * m * n
    out = ops.fp8_gemm_blockwise(xq, wq, xs, ws)
    _within_bounds(out, xq, wq, xs, ws, need // (4 * m * n))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = ops.fp8_gemm_blockwise(xq, wq, xs, ws)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, out)
    # one row fewer of the workspace: the best plan that fits; none: one piece
    short = torch.empty(need // 4 - m * n, device=gpu_device)
    for space in (short, None):
        got = torch.zeros_like(out)
        _lib.check(_call(xq, wq, xs, ws, got, space, -1), "gemm_ws")
        _within_bounds(got, xq, wq, xs, ws, 16)


# Shapes of up to 256 rows that the streaming forms run without a workspace, in parts with one. Those take every factor as it is, and
# so do the parts: blocks of zeros in both operands (whose factors a quantiser makes very small) among large ones, a factor
# of zero beside codes that are none and small factors, neighbours up to 2^120 apart, factors of either sign.
@pytest.mark.parametrize("m,n,k", [(32, 1024, 28672), (92, 515, 26368), (33, 1100, 28656)])
@pytest.mark.parametrize("factors", ["zero blocks", "zero factors", "far apart", "signs"])
def test_parts_take_any_factors(gpu_device, m, n, k, factors):
    print(f"case {m}x{n}x{k} {factors}", flush=True)
    xq, wq, xs, ws = _inputs(m, n, k, gpu_device, seed=1)
    gk = xs.shape[1]
    if factors == "zero blocks":
        xs *= 2.0**20
        ws *= 2.0**20
        for kb in (1, 5, 6, 40, gk - 1):
            xq[:, kb * 128 : (kb + 1) * 128] = 0
            wq[:, kb * 128 : (kb + 1) * 128] = 0
            xs[:, kb] = 1e-12 / 448
            ws[:, kb] = 1e-12 / 448
    elif factors == "zero factors":
        xs *= 2.0**-40
        ws *= 2.0**-40
        for kb in (0, 7, 30, 31, gk - 1):
            xs[:, kb] = 0.0
    elif factors == "far apart":
        xs[:, ::2] *= 2.0**60
        xs[:, 1::2] *= 2.0**-60
    else:
        xs *= torch.where(torch.rand(xs.shape, device=gpu_device) < 0.5, -1.0, 1.0)
        ws *= torch.where(torch.rand(ws.shape, device=gpu_device) < 0.5, -1.0, 1.0)
    parts = _lib.load().mi355x_fp8_blockwise_workspace_bytes(m, n, k) // (4 * m * n)
    assert parts >= 2
    _within_bounds(ops.fp8_gemm_blockwise(xq, wq, xs, ws), xq, wq, xs, ws, parts)
    streaming = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
    _lib.check(_call(xq, wq, xs, ws, streaming, None, _lib.BLOCK_ONE_TILE if m <= 64 else _lib.BLOCK_NARROW), "gemm_ws")
    _within_bounds(streaming, xq, wq, xs, ws, 1)


def test_factors_without_their_workspace_are_refused(gpu_device):
    xq, wq, xs, ws = _inputs(128, 128, 1024, gpu_device)
    out = torch.zeros((128, 128), dtype=torch.bfloat16, device=gpu_device)
    space = torch.empty(3 * 128 * 128, device=gpu_device)
    for form, given in ((_lib.BLOCK_TILES_128 + 256 * 4, space), (_lib.BLOCK_TILES_128 + 256 * 2, None), (_lib.BLOCK_TILES_256 + 256 * 2, space)):
        assert _call(xq, wq, xs, ws, out, given, form) == _lib.EINVAL
    assert _call(xq, wq, xs, ws, out, space.view(torch.uint8)[4:].view(torch.float32), _lib.BLOCK_TILES_128 + 256 * 2) == _lib.EINVAL
