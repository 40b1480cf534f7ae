"""The block-scaled form that keeps A on chip (up to 16 rows, one or two 16-row tiles of B a CU, a wave's K steps 16 apart), at the edges of
its tiles, rounds of steps and K, against float64. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import ops
from tritonbench_amd._lib import BLOCK_RESIDENT

from test_gpu_blockwise_forms import _check, _expand, _run

pytestmark = pytest.mark.gpu

# one tile, tiles for some CUs, one each, one more than that, two each but for one CU, two each; one to four rounds of steps, whole and with a
# last step that is partial; tiles of either side of a scale block's edge in one workgroup
@pytest.mark.parametrize("m,n,k", [(1, 16, 8192), (16, 144, 8192), (9, 160, 6160), (16, 2048, 2000), (16, 1552, 3088), (13, 4112, 3984),
                                   (16, 4240, 2000), (7, 2784, 5456), (16, 8176, 2048), (16, 8192, 2048), (16, 8176, 4096), (16, 8192, 8192),
                                   (9, 8192, 8176)])
def test_against_float64(gpu_device, m, n, k):
    print(f"case m={m} n={n} k={k}", flush=True)
    _check(m, n, k, gpu_device, BLOCK_RESIDENT)


@pytest.mark.parametrize("side", ["a", "b"])
@pytest.mark.parametrize("m,n,k", [(16, 144, 8192), (9, 160, 6160), (16, 4240, 2000), (16, 8192, 8192)])
def test_an_infinite_factor_of_the_last_block(gpu_device, m, n, k, side):
    one = torch.ones(1, device=gpu_device).to(torch.float8_e4m3fn)
    xq, wq = one.expand(m * k).clone().view(m, k), one.expand(n * k).clone().view(n, k)
    xs, ws = (torch.ones((-(-r // 128), -(-k // 128)), device=gpu_device) for r in (m, n))
    (xs if side == "a" else ws)[0, -1] = float("inf")
    want = torch.full((m, n), float(k), dtype=torch.float64, device=gpu_device)
    want[:, slice(None) if side == "a" else slice(0, 128)] = float("inf")
    got = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
    assert torch.equal(_run(xq, wq, xs, ws, got, BLOCK_RESIDENT), want.to(torch.bfloat16))


# rows of C on any 2 bytes, factors 2^120 apart between neighbouring blocks and of zero; a replay of the library's choice, which is this form
def test_odd_rows_of_c_any_factors_and_capture(gpu_device):
    m, n, k = 11, 8000, 6000
    g = torch.Generator(device=gpu_device).manual_seed(5)
    xq, wq = (torch.randn((r, k), generator=g, device=gpu_device).to(torch.float8_e4m3fn) for r in (m, n))
    xs, ws = (torch.rand((-(-r // 128), -(-k // 128)), generator=g, device=gpu_device) + 0.5 for r in (m, n))
    xs[:, ::2] *= 2.0**60
    xs[:, 1::2] *= 2.0**-60
    xs[:, 3] = 0.0
    canvas = torch.full((m + 2, n + 5), 7.0, dtype=torch.bfloat16, device=gpu_device)
    out = canvas[1:-1, 3:-2]
    _run(xq, wq, xs, ws, out, BLOCK_RESIDENT)
    exact = _expand(xq, xs) @ _expand(wq, ws).t()
    assert ((out.double() - exact).norm() / exact.norm()).item() < 2.0**-8  # (one rounding to bf16)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = ops.fp8_gemm_blockwise(xq, wq, xs, ws)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, out)
    out.fill_(7.0)
    assert (canvas == 7.0).all()
