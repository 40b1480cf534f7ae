"""The second pass of a split-K launch at the edges of its forms: one row a thread up to 2048 workgroups, four rows above
where N is a multiple of 4. Integer codes and power-of-two scales: every partial sum is exact in f32 and the result is the
float64 one rounded once, bit for bit. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu


# 1024 x 2048 is the last of the one-row form; then a remainder of 1, 3 and 0 rows, N a multiple of 4 but not of 8, N off it
@pytest.mark.parametrize("m,n", [(1024, 2048), (1025, 2048), (1027, 2052), (516, 8196), (1, 4), (1029, 2051), (5, 524292)])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 9])
@pytest.mark.parametrize("bias,out_type,pad", [(False, torch.bfloat16, 0), (True, torch.float16, 4), (True, torch.bfloat16, 3)])
def test_second_pass_bit_for_bit(gpu_device, m, n, splits, bias, out_type, pad):
    print(f"case m={m} n={n} splits={splits} bias={bias} {out_type} pad={pad}", flush=True)
    k = 9 * 128
    gen = torch.Generator(device=gpu_device).manual_seed(m + n)
    ints = lambda *s: torch.randint(-2, 3, s, generator=gen, device=gpu_device).to(torch.float32)
    powers = lambda s: 2.0 ** torch.randint(-3, 4, (s,), generator=gen, device=gpu_device).to(torch.float32)
    x, w, xs, ws = ints(m, k), ints(n, k), powers(m), powers(n)
    b = ints(n).to(torch.bfloat16) if bias else None
    # (f32 holds every sum of products, its scaled value and that plus the bias exactly)
    want = (x @ w.T) * xs[:, None] * ws[None, :]
    want = (want + b.float()[None, :] if bias else want).to(out_type)
    canvas = torch.full((m + 1, n + pad), -77.0, dtype=out_type, device=gpu_device)
    ops.fp8_gemm_rowwise(x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), xs, ws, bias=b, out=canvas[:m, :n],
                         variant=_lib.tiled_variant(1, splits), out_dtype=out_type)
    assert torch.equal(canvas[:m, :n], want)
    assert torch.all(canvas[m:] == -77.0) and torch.all(canvas[:, n:] == -77.0)
