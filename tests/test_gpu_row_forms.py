"""Every way in which a row's chunks are dealt out over lanes and rounds (by the number of rows and the row's length), at its edges:
the longest row of a form and the shortest of the next, with as many rows as choose the form. The first rows of a call against the
oracle, and all its rows, equal to those by construction, against them. A row with a NaN or an infinity takes a path of its own."""
import pytest
import torch

from oracle import fp8_rowwise as orc
from tritonbench_amd import ops

from test_gpu_fused_quant import _check_codes

pytestmark = pytest.mark.gpu

ROWS = [2, 257, 2049]  # few, some and many: a row a CU, up to 2048
CHUNKS = [63, 65, 128, 129, 192, 193, 256, 257, 384, 385, 512, 513, 768, 769, 1024, 1025, 1280, 1281, 1537, 2049, 2561, 3073, 3585, 4095, 4097]


def _repeated(x, rows):
    return x.repeat(-(-rows // x.shape[0]), 1)[:rows].contiguous()


def _same_rows(t, period):
    bits = t.view(torch.uint8) if t.dtype != torch.float32 else t.view(torch.int32)
    return all(torch.equal(bits[i::period], bits[i : i + 1].expand(bits[i::period].shape)) for i in range(period))


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("source", [torch.bfloat16, torch.float32])
def test_quantiser(gpu_device, rows, source):
    for chunks in CHUNKS + ([7168, 7169] if source == torch.float32 else []):
        k = chunks * 16 // source.itemsize
        k += -k % 16  # (whole 16-byte chunks of codes too: the longest row of a form stays what it is)
        assert chunks % 2 or k * source.itemsize == chunks * 16
        print(f"case {rows}x{k} {source}", flush=True)
        x = torch.randn((4, k), generator=torch.Generator().manual_seed(k)).to(source)
        x[1, k - 1], x[2, 0], x[3, k // 2] = 300.0, float("nan"), float("-inf")  # (the first two rows' largest wherever they fall)
        want_q, want_s = orc.fp8_row_quantize(x)
        got_q, got_s = ops.fp8_row_quantize(_repeated(x, rows).to(gpu_device))
        n = min(rows, 4)
        got, want = got_q[:n].view(torch.uint8).cpu(), want_q[:n].view(torch.uint8)
        assert torch.equal(got, want.where((want & 0x7F) != 0x7F, got | 0x7F))  # (a NaN of either sign)
        assert torch.equal(got_s[:n].cpu().nan_to_num(nan=-1.0), want_s[:n].float().nan_to_num(nan=-1.0))
        assert _same_rows(got_q, 4) and _same_rows(got_s[:, None], 4)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("front", ["rms_norm", "silu_mul"])
def test_fused_front_ends(gpu_device, rows, front):
    for chunks in CHUNKS:
        k = chunks * 8
        k += -k % 16
        print(f"case {front} {rows}x{k}", flush=True)
        x1, x2, _, _, wd = orc.make_fused_inputs(2, 16, k)
        if front == "rms_norm":
            # Scaled values that lie between two codes in real arithmetic go either way. With a row's largest value 161/32 * 129/128 they are
            # those of products that are multiples of 3 * 23 * 43: next to none.
            x1, wd = x1.clamp(-3.5, 3.5), wd.clamp(0.5, 1.25)
            x1[0, k // 3], x1[1, k // 3], wd[k // 3] = 161 / 32, -161 / 32, 129 / 128
        if front == "rms_norm":
            want_q, want_s = orc.rms_norm_fp8_rowwise_quant(x1, wd)
            got_q, got_s = ops.rms_norm_fp8_rowwise_quant(_repeated(x1, rows).to(gpu_device), wd.to(gpu_device))
        else:
            want_q, want_s = orc.silu_mul_fp8_rowwise_quant(x1, x2)
            got_q, got_s = ops.silu_mul_fp8_rowwise_quant(_repeated(x1, rows).to(gpu_device), _repeated(x2, rows).to(gpu_device))
        _check_codes(got_q[:2], got_s[:2], want_q, want_s)
        assert _same_rows(got_q, 2) and _same_rows(got_s[:, None], 2)
