"""Rows of B that start off the 128-byte lines: the instances without the streaming policy, on both sides of the rules that choose them.
The kernels sum in the same order with and without the policy, so rows padded by 16 bytes, or by half a line, give the bits that rows on the lines give."""
import numpy as np
import pytest
import torch

from tritonbench_amd import _lib

pytestmark = pytest.mark.gpu

ONE_TILE, NARROW, RESIDENT = (_lib.VARIANT_SKINNY | pin for pin in (_lib.SKINNY_ONE_TILE, _lib.SKINNY_NARROW, _lib.SKINNY_RESIDENT))


def _operands(m, n, k, dev):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    codes = lambda r: torch.randn((r, k), generator=g, device=dev, dtype=torch.bfloat16).to(torch.float8_e4m3fn)
    return codes(m), codes(n), g


def _padded(w, pad):
    wide = torch.full((w.shape[0], w.shape[1] + pad), 0x7F, dtype=torch.uint8, device=w.device)  # (NaN codes past the rows' ends)
    wide[:, : w.shape[1]] = w.view(torch.uint8)
    return wide.view(torch.float8_e4m3fn)[:, : w.shape[1]]


def _same_and_right(run, xq, wq, exact):
    bits = []
    for w in (wq, _padded(wq, 16), _padded(wq, 64)):
        out = torch.full((xq.shape[0], wq.shape[0]), float("nan"), dtype=torch.bfloat16, device=xq.device)
        run(w, out)
        torch.cuda.synchronize()
        assert ((out.double() - exact).norm() / exact.norm()).item() < 2.0**-8  # (one rounding to bf16)
        bits.append(out.view(torch.int16).cpu().numpy())
    assert np.array_equal(bits[0], bits[1]) and np.array_equal(bits[0], bits[2])


ROW_CASES = [
    # eight steps and nine, panels of 1.5 MB and more, each of the row counts
    *[(ONE_TILE, m, n, k, False) for m in (1, 17, 40, 64) for n, k in ((1540, 1024), (1540, 1152), (1364, 1152), (1366, 1152))],
    # tiles of 8, 12, 16 and 20 columns, rows on both sides of the rule's, two row blocks
    *[(NARROW, m, n, 1152, False) for m in (8, 9, 32, 33) for n in (2048, 2052, 4096, 4100)],
    *[(NARROW, 100, n, k, False) for n, k in ((400, 1024), (401, 1024), (2000, 1152))],
    *[(RESIDENT, m, n, k, m == 3) for m in (3, 16) for n, k in ((1600, 1024), (1600, 1152), (528, 1152))],
    # tiles of one and two tile rows whose launch streams B, the kernels for a K tail without one
    *[(_lib.tiled_variant(c, s), 200, 1000, 1152, s == 1) for c in range(_lib.NUM_TILE_CONFIGS) for s in (1, 3)],
    (_lib.tiled_variant(0, 3), 64, 1001, 1024, False),
]


@pytest.mark.parametrize("variant,m,n,k,with_bias", ROW_CASES)
def test_row_scaled(gpu_device, variant, m, n, k, with_bias):
    print(f"case variant {variant:#x} {m}x{n}x{k} bias={with_bias}", flush=True)
    lib = _lib.load()
    xq, wq, g = _operands(m, n, k, gpu_device)
    xs, ws = (torch.rand(r, generator=g, device=gpu_device) + 0.5 for r in (m, n))
    bias = torch.randn(n, generator=g, device=gpu_device).to(torch.bfloat16) if with_bias else None
    need = lib.mi355x_fp8_rowwise_workspace_bytes(m, n, k, variant)
    space = torch.full((need // 4 + 4,), float("nan"), device=gpu_device)
    exact = (xq.double() @ wq.double().t()) * xs.double()[:, None] * ws.double()[None, :] + (bias.double() if with_bias else 0.0)

    def run(w, out):
        _lib.check(lib.mi355x_fp8_rowwise_gemm(xq.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), bias.data_ptr() if with_bias else None,
                                               out.data_ptr(), m, n, k, k, w.stride(0), n, space.data_ptr(), need, variant,
                                               torch.cuda.current_stream().cuda_stream), "gemm")

    _same_and_right(run, xq, wq, exact)


@pytest.mark.parametrize("form,m,n,k", [*[(_lib.BLOCK_ONE_TILE, m, n, k) for m in (1, 64) for n, k in ((1540, 1024), (1540, 1152), (520, 1152))],
                                        *[(_lib.BLOCK_NARROW, m, n, 1152) for m in (16, 17) for n in (2048, 5120, 5124)],
                                        (_lib.BLOCK_NARROW, 100, 512, 1024), (_lib.BLOCK_TILES_128, 100, 1000, 1152),
                                        (_lib.BLOCK_TILES_128_STREAM, 100, 1000, 1152), (_lib.BLOCK_TILES_256, 100, 1000, 1152)])
def test_block_scaled(gpu_device, form, m, n, k):
    print(f"case form {form} {m}x{n}x{k}", flush=True)
    lib = _lib.load()
    xq, wq, g = _operands(m, n, k, gpu_device)
    xs, ws = (torch.rand((-(-r // 128), -(-k // 128)), generator=g, device=gpu_device) + 0.5 for r in (m, n))
    each = lambda q, s: q.double() * s.double().repeat_interleave(128, 0)[: q.shape[0]].repeat_interleave(128, 1)[:, :k]
    exact = each(xq, xs) @ each(wq, ws).t()

    def run(w, out):
        _lib.check(lib.mi355x_fp8_blockwise_gemm_ex(xq.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), out.data_ptr(), m, n, k, k,
                                                    w.stride(0), n, form, torch.cuda.current_stream().cuda_stream), "blockwise_gemm_ex")

    _same_and_right(run, xq, wq, exact)
