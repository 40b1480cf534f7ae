"""128x128 tiles with the deep ring on rows off the 128-byte lines, which are fetched in whole lines from the line that each begins in: the
bits of the same rows on the lines, whatever lies around them. Pinned, at most one work item a workgroup."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _codes(rows, k, pitch, shift, fill, dev, seed):
    """[rows, k] codes, row r from byte shift + r * pitch of a buffer (on 256 bytes) that is `fill` everywhere else."""
    codes = torch.randn((rows, k), generator=torch.Generator(device=dev).manual_seed(seed), device=dev).to(torch.float8_e4m3fn)
    buffer = torch.full((shift + rows * pitch + 128,), fill, dtype=torch.uint8, device=dev)
    view = buffer[shift : shift + rows * pitch].view(rows, pitch)[:, :k]
    view.copy_(codes.view(torch.uint8))
    return view.view(torch.float8_e4m3fn)


# twelve steps, from which on the windows are used, with a last one of one chunk, of seven and whole; with K on the steps the pitch alone is off the
# lines. Three parts: whole ones, and a last one that is shorter and has the partial step
@pytest.mark.parametrize("k,splits", [(1424, 1), (1520, 1), (1536, 1), (1552, 1), (2032, 1), (4112, 1), (4608, 3), (4624, 3), (4848, 3)])
@pytest.mark.parametrize("m,n", [(1, 1), (128, 128), (129, 300), (400, 3000)])
def test_the_bits_of_rows_on_the_lines(gpu_device, k, m, n, splits):
    variant = _lib.tiled_variant(6, splits)
    xs, ws = (torch.rand(r, generator=torch.Generator(device=gpu_device).manual_seed(r), device=gpu_device) + 0.5 for r in (m, n))
    bias = torch.randn(n, device=gpu_device).to(torch.bfloat16) if m > 128 else None
    on = -(-k // 128) * 128
    want = ops.fp8_gemm_rowwise(_codes(m, k, on, 0, 0x7F, gpu_device, 1), _codes(n, k, on, 0, 0x7F, gpu_device, 2), xs, ws, bias=bias, variant=variant)
    # (pitch past K, first byte) of either operand: NaN codes around the rows
    for (pa, sa), (pb, sb) in (((16, 0), (0, 16)), ((80, 48), (0, 0)), ((0, 0), (112, 112)), ((48, 96), (32, 64)), ((0, 16), (96, 0))):
        print(f"case {m}x{n}x{k} splits={splits} a +{pa} at {sa}, b +{pb} at {sb}", flush=True)
        x, w = _codes(m, k, k + pa, sa, 0x7F, gpu_device, 1), _codes(n, k, k + pb, sb, 0x7F, gpu_device, 2)
        canvas = torch.full((m + 2, n + 3), 7.0, dtype=torch.bfloat16, device=gpu_device)
        out = ops.fp8_gemm_rowwise(x, w, xs, ws, bias=bias, out=canvas[1:-1, 1:-2], variant=variant)
        assert torch.equal(out, want)
        out.fill_(7.0)
        assert (canvas == 7.0).all()
