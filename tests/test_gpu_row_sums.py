"""The fused RMSNorm's sum of squares is added up in an order that hangs on the row's length alone: the codes and scales of a row, bit for
bit, as that order gives them in f32, with as many rows as choose each form of the kernel. Needs an MI355X."""
import numpy as np
import pytest
import torch

from oracle import fp8_rowwise as orc
from tritonbench_amd import ops

from test_gpu_row_forms import _repeated, _same_rows

pytestmark = pytest.mark.gpu

# rows of 16-byte chunks on both sides of each line of the order and of the forms
CHUNKS = [2, 64, 66, 128, 130, 192, 194, 256, 258, 512, 514, 768, 770, 1024, 1026, 1280, 1282, 1536, 1538, 2048, 2050, 2560, 2562, 3072, 3074, 3584, 3586, 4096, 4098, 8192, 8194]


def _sum_of_squares(x):
    """x [rows, chunks, 8] f32 from bf16, whose squares f32 holds exactly: a multiply-add rounds as the addition of one does."""
    rows, chunks, _ = x.shape
    lanes = 64 if chunks <= 256 else 256 if chunks <= 1024 else 512 if chunks <= 4096 else 1024
    padded = np.zeros((rows, -(-chunks // lanes) * lanes, 8), dtype=np.float32)
    padded[:, :chunks] = x
    chains = np.zeros((rows, lanes), dtype=np.float32)
    for turn in padded.reshape(rows, -1, lanes, 8).transpose(1, 3, 0, 2).reshape(-1, rows, lanes):
        chains += turn * turn
    groups = chains.reshape(rows, -1, 64)
    for bit in (32, 16, 8, 4, 2, 1):
        groups = groups[..., :bit] + groups[..., bit:]
    total = groups[:, 0, 0].copy()
    for g in range(1, groups.shape[1]):
        total += groups[:, g, 0]
    return total


@pytest.mark.parametrize("rows", [1, 2, 257, 2049])
def test_a_row_alone_and_among_others(gpu_device, rows):
    for chunks in CHUNKS:
        k = chunks * 8
        print(f"case {rows}x{k}", flush=True)
        x, _, _, _, weight = orc.make_fused_inputs(3, 16, k, seed_tag=5)
        eps = np.float32(1e-5)
        f = x.float().numpy()
        rstd = np.float32(1) / np.sqrt(_sum_of_squares(f.reshape(3, chunks, 8)) / np.float32(k) + eps)
        want_q, want_s = orc.fp8_row_quantize(torch.from_numpy((f * rstd[:, None]) * weight.float().numpy()))
        got_q, got_s = ops.rms_norm_fp8_rowwise_quant(_repeated(x, rows).to(gpu_device), weight.to(gpu_device), float(eps))
        n = min(rows, 3)
        assert torch.equal(got_s[:n].cpu().flatten(), want_s[:n].float().flatten())
        assert torch.equal(got_q[:n].view(torch.uint8).cpu(), want_q[:n].view(torch.uint8))
        assert _same_rows(got_q, n) and _same_rows(got_s.reshape(rows, 1), n)
