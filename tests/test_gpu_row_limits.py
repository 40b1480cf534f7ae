"""More rows than one launch of the quantiser or a fused front end holds (fewer than 2^32 lanes): 256 lanes a row from 16777213 rows on, a
wave each from 67108861 on. Needs an MI355X and, for the former, 110 GB of its memory."""
import pytest
import torch

from oracle import fp8_rowwise as orc
from tritonbench_amd import ops

pytestmark = pytest.mark.gpu

PERIOD = 8191  # (rows that differ: where a launch begins is no multiple of it)


def _run(rows, k, need, front, dev):
    if torch.cuda.mem_get_info(dev)[0] < need:
        pytest.skip(f"needs {need >> 30} GB of device memory")
    print(f"case {front} {rows}x{k}", flush=True)
    block = torch.randn((PERIOD, k), generator=torch.Generator().manual_seed(k)).to(torch.bfloat16)
    weight = torch.ones(k, dtype=torch.bfloat16)
    x = torch.empty((rows, k), dtype=torch.bfloat16, device=dev)
    for r in range(0, rows, PERIOD):
        x[r : r + PERIOD] = block[: rows - r].to(dev) if r == 0 else x[: min(PERIOD, rows - r)]
    call = {"quantise": ops.fp8_row_quantize, "rms_norm": lambda t: ops.rms_norm_fp8_rowwise_quant(t, weight.to(dev)),
            "silu_mul": lambda t: ops.silu_mul_fp8_rowwise_quant(t, t)}[front]
    q, s = call(x)
    few_q, few_s = call(x[:PERIOD])
    if front == "quantise":
        want_q, want_s = orc.fp8_row_quantize(block[:64])
        assert torch.equal(few_q[:64].view(torch.uint8).cpu(), want_q.view(torch.uint8)) and torch.equal(few_s[:64].cpu(), want_s.float())
    wrong = torch.zeros((), dtype=torch.int64, device=dev)
    for r in range(0, rows, PERIOD):
        n = min(PERIOD, rows - r)
        wrong += (q[r : r + n].view(torch.uint8) != few_q[:n].view(torch.uint8)).sum() + (s[r : r + n] != few_s[:n]).sum()
    assert wrong.item() == 0


@pytest.fixture(autouse=True)
def memory_back():
    yield
    torch.cuda.empty_cache()


@pytest.mark.parametrize("front", ["quantise", "rms_norm", "silu_mul"])
def test_256_lanes_a_row(gpu_device, front):
    _run((1 << 24) + 5, 2064, 130 << 30, front, gpu_device)


@pytest.mark.parametrize("front", ["quantise", "rms_norm", "silu_mul"])
def test_a_wave_a_row(gpu_device, front):
    _run((1 << 26) + 5, 16, 8 << 30, front, gpu_device)
