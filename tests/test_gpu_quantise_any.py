"""The row quantiser on rows that start at any element and end anywhere, bit for bit against the oracle: every form's edges,
rows of one chunk and a little more, sources and results off the 16-byte boundary, NaN and infinities. Needs an MI355X."""
import pytest
import torch

from oracle import fp8_rowwise as orc
from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


def _source(dtype, rows, cols, lead, pad):
    buf = orc.randn_f32(rows, lead + cols + pad, 1.0, seed=cols).to(dtype)
    return buf, buf[:, lead:lead + cols]


def _same(got, want):
    q, inv = got
    wq, winv = want
    assert torch.equal(q.cpu().view(torch.uint8), wq.view(torch.uint8))
    assert torch.equal(inv.cpu().view(torch.int32), winv.view(torch.int32))


# (columns around one chunk, the whole rounds of a wave and of 256, 512 and 1024 lanes, and past the registers of each)
@pytest.mark.parametrize("dtype,rows,cols", [
    (F32, 3, 1), (F32, 3, 3), (F32, 3, 4), (F32, 3, 5), (F32, 5, 1041), (F32, 5, 4095), (F32, 5, 4096), (F32, 3, 4097),
    (F32, 2, 16385), (F32, 2, 40001), (F32, 2051, 17), (F32, 2050, 511), (F32, 2049, 2047),
    (BF16, 3, 1), (BF16, 3, 7), (BF16, 3, 8), (BF16, 3, 9), (BF16, 5, 1041), (BF16, 5, 8191), (BF16, 5, 8192), (BF16, 3, 8193),
    (BF16, 2, 32771), (BF16, 2, 70001), (BF16, 2051, 33), (BF16, 2050, 1023), (BF16, 2049, 4095),
    # a wave each with one or two rounds of loads, and the element-by-element kernel for few short bf16 rows
    (F32, 7, 63), (F32, 7, 255), (F32, 7, 256), (F32, 7, 257), (F32, 2049, 255), (BF16, 5, 256), (BF16, 5, 257), (BF16, 513, 66),
    (BF16, 2048, 63), (BF16, 514, 511), (BF16, 6, 512), (BF16, 6, 513), (BF16, 2049, 1023), (BF16, 2049, 1025),
])
@pytest.mark.parametrize("lead,pad", [(0, 0), (1, 2)])
def test_rows_that_start_anywhere(gpu_device, dtype, rows, cols, lead, pad):
    buf, x = _source(dtype, rows, cols, lead, pad)
    _same(ops.fp8_row_quantize(buf.to(gpu_device)[:, lead:lead + cols]), orc.fp8_row_quantize(x.contiguous()))


@pytest.mark.parametrize("dtype,cols", [(F32, 1041), (BF16, 2051), (BF16, 64)])
def test_results_that_start_anywhere_leave_the_rest_alone(gpu_device, dtype, cols):
    rows, pitch, lead = 9, cols + 13, 5
    _, x = _source(dtype, rows, cols, 0, 0)
    want_q, want_inv = orc.fp8_row_quantize(x)
    d = x.to(gpu_device)
    q = torch.full((rows * pitch + lead,), 0x55, dtype=torch.uint8, device=gpu_device)
    inv = torch.empty(rows, device=gpu_device)
    ops.fp8_row_quantize(d)
    st = _lib.load().mi355x_fp8_rowwise_quantize(d.data_ptr(), _lib.SRC_F32 if dtype == F32 else _lib.SRC_BF16, q.data_ptr() + lead,
                                                 inv.data_ptr(), rows, cols, d.stride(0), pitch,
                                                 torch.cuda.current_stream().cuda_stream)
    _lib.check(st, "quantize")
    got = q.cpu()[lead:].view(rows, pitch)
    _same((got[:, :cols].contiguous().view(torch.float8_e4m3fn), inv), (want_q, want_inv))
    assert torch.all(got[:, cols:] == 0x55) and torch.all(q.cpu()[:lead] == 0x55)


@pytest.mark.parametrize("dtype,cols", [(F32, 1041), (BF16, 1041), (BF16, 8199), (F32, 101), (BF16, 301), (BF16, 101)])
def test_non_finite_and_zero_rows(gpu_device, dtype, cols):
    _, x = _source(dtype, 5, cols, 0, 0)
    x = x.clone()
    x[0, cols - 1] = float("nan")
    x[1, cols - 1] = float("inf")
    x[2, cols - 2] = float("-inf")
    x[3] = 0
    want_q, want_inv = orc.fp8_row_quantize(x)
    q, inv = ops.fp8_row_quantize(x.to(gpu_device))
    got, want = q.cpu().view(torch.uint8), want_q.view(torch.uint8)
    nan = (want & 0x7F) == 0x7F
    assert torch.equal((got & 0x7F) == 0x7F, nan) and torch.equal(got[~nan], want[~nan])
    assert torch.equal(inv.cpu().isnan(), want_inv.isnan()) and torch.equal(inv.cpu()[~want_inv.isnan()], want_inv[~want_inv.isnan()])
