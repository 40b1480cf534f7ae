"""Results that the native binding allocates: the same kind of tensor, and seen by whoever watches, whichever way they were made."""
import ctypes

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tritonbench_amd import ops

pytestmark = pytest.mark.gpu


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _calls(x, w):
    xq, xs = ops.fp8_row_quantize(x)
    wq, ws = ops.fp8_row_quantize(w)
    return [xq, xs, ops.fp8_gemm_rowwise(xq, wq, xs, ws)]


def test_results_are_the_same_whoever_watches(gpu_device):
    x, w = (torch.randn((r, 512), device=gpu_device, dtype=torch.bfloat16) for r in (5, 48))
    plain = _calls(x, w)
    with torch.inference_mode():
        inference = _calls(x, w)
    with _Seen() as seen:
        watched = _calls(x, w)
    with torch.autocast("cuda"):
        cast = _calls(x, w)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        profiled = _calls(x, w)
    assert sum("aten.empty" in n for n in seen.names) >= 5
    assert sum(e.count for e in prof.key_averages() if e.key == "aten::empty") >= 5
    assert all(t.is_inference() for t in inference) and not any(t.is_inference() for t in plain)
    for other in (inference, watched, cast, profiled):
        for a, b in zip(plain, other):
            assert (a.dtype, a.shape, a.stride(), a.device, a.requires_grad) == (b.dtype, b.shape, b.stride(), b.device, b.requires_grad)
            assert torch.equal(a.view(torch.uint8) if a.dtype == torch.float8_e4m3fn else a, b.view(torch.uint8) if b.dtype == torch.float8_e4m3fn else b)
    # tensors like any other: a version of their own, room for a gradient, an allocation of their own that is given back
    out = plain[2]
    version = out._version
    out.add_(1)
    assert out._version == version + 1 and out.clone().requires_grad_().requires_grad
    assert len({t.untyped_storage().data_ptr() for t in plain}) == 3
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(gpu_device)
    more = _calls(x, w)
    assert torch.cuda.memory_allocated(gpu_device) > before
    del more
    assert torch.cuda.memory_allocated(gpu_device) == before


def _nodes(call):
    """What a captured call consists of: its launches and whatever its allocations add."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    count = ctypes.c_size_t()
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


def test_new_memory_is_filled_where_that_is_asked_for(gpu_device):
    x = torch.randn((5, 512), device=gpu_device, dtype=torch.bfloat16)
    plain = ops.fp8_row_quantize(x)
    alone = _nodes(lambda: ops.fp8_row_quantize(x))
    try:
        torch.use_deterministic_algorithms(True)
        filled = _nodes(lambda: ops.fp8_row_quantize(x))
        other = ops.fp8_row_quantize(x)
        torch.utils.deterministic.fill_uninitialized_memory = False
        not_filled = _nodes(lambda: ops.fp8_row_quantize(x))
    finally:
        torch.use_deterministic_algorithms(False)
        torch.utils.deterministic.fill_uninitialized_memory = True
    assert filled >= alone + 2 and not_filled == alone  # (codes and scales)
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(plain, other))
