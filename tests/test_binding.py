"""The native binding against the wrappers' own path through ctypes: the same results, and None for what is theirs."""
import pytest
import torch

from tritonbench_amd import _lib, ops

FP8 = torch.float8_e4m3fn


class _Refuses:
    def __getattr__(self, name):
        return lambda *args: None


def _codes(*shape):
    return torch.randint(-3, 4, shape).to(torch.float32).to(FP8)


def _calls(dev):
    """name -> call without outputs of its own"""
    x, w, xs, ws = (t.to(dev) for t in (_codes(40, 272), _codes(96, 272), torch.rand(40) + 0.5, torch.rand(96) + 0.5))
    bias, space = torch.randn(96, device=dev, dtype=torch.bfloat16), torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    sizes = torch.tensor([13, 0, 20], dtype=torch.int32, device=dev)
    bx, bw = torch.rand(1, 3, device=dev) + 0.5, torch.rand(1, 3, device=dev) + 0.5
    h, g = torch.randn(33, 256, device=dev, dtype=torch.bfloat16), torch.randn(33, 256, device=dev, dtype=torch.bfloat16)
    out = torch.zeros(40, 100, device=dev, dtype=torch.bfloat16)
    return {
        "row": lambda: ops.fp8_gemm_rowwise(x, w, xs, ws),
        "row, every option": lambda: ops.fp8_gemm_rowwise(x, w, xs, ws, bias=bias, out=out[:, :96], variant=_lib.VARIANT_TILED,
                                                          workspace=space),
        "row, float16": lambda: ops.fp8_gemm_rowwise(x, w, xs, ws, bias=bias, out_dtype=torch.float16),
        "row, any K": lambda: ops.fp8_gemm_rowwise(x[:, 1:], w[:, 1:], xs, ws),
        "grouped": lambda: ops.fp8_gemm_rowwise_grouped(x, w, sizes, xs, ws),
        "block": lambda: ops.fp8_gemm_blockwise(x, w, bx, bw),
        "quantise": lambda: ops.fp8_row_quantize(h),
        "quantise, fp32": lambda: ops.fp8_row_quantize(h.float()[:, 3:]),
        "block quantise": lambda: ops.fp8_block_quantize(h),
        "RMSNorm": lambda: ops.rms_norm_fp8_rowwise_quant(h, g[0], 1e-6),
        "SiLU-mul": lambda: ops.silu_mul_fp8_rowwise_quant(h, g),
    }


def _bits(result):
    return [t.contiguous().view(torch.uint8).clone() for t in (result if isinstance(result, tuple) else (result,))]


@pytest.mark.gpu
def test_both_ways_give_the_same_bits(gpu_device, monkeypatch):
    for name, call in _calls(gpu_device).items():
        call()  # (the first call on a device sets it up the long way)
        native = call()
        shapes = [(t.shape, t.stride(), t.dtype, t.device) for t in (native if isinstance(native, tuple) else (native,))]
        native = _bits(native)
        with monkeypatch.context() as m:
            m.setattr(_lib, "binding", lambda: _Refuses())
            own = call()
        assert shapes == [(t.shape, t.stride(), t.dtype, t.device) for t in (own if isinstance(own, tuple) else (own,))], name
        assert all(torch.equal(a, b) for a, b in zip(native, _bits(own))), name


@pytest.mark.gpu
def test_the_call_goes_to_the_current_stream_and_out_comes_back_itself(gpu_device):
    calls = _calls(gpu_device)
    want = _bits(calls["row"]())
    calls["row, every option"]()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):  # (raises if anything went to another stream)
            got = calls["row"]()
        graph.replay()
        stream.synchronize()
    assert torch.equal(_bits(got)[0], want[0])
    out = torch.empty(40, 96, device=gpu_device, dtype=torch.bfloat16)
    x, w, s = _codes(40, 256).to(gpu_device), _codes(96, 256).to(gpu_device), torch.ones(96, device=gpu_device)
    assert ops.fp8_gemm_rowwise(x, w, s[:40], s, out=out) is out


@pytest.mark.gpu
def test_what_is_wrong_with_a_call_is_left_to_the_wrappers(gpu_device):
    b = _lib.binding()
    x, w, s = _codes(8, 256).to(gpu_device), _codes(16, 256).to(gpu_device), torch.ones(16, device=gpu_device)
    ops.fp8_gemm_rowwise(x, w, s[:8], s)
    good = [x, w, s[:8], s, None, None, 0, None, False]
    assert b.gemm_rowwise(*good) is not None

    class Sub(torch.Tensor):
        pass

    for at, bad in ((0, x.float()), (0, x[0]), (0, x.t()), (0, x[:, :128]), (0, x.as_subclass(Sub)), (1, w.cpu()), (1, None),
                    (2, s), (2, s[:16:2]), (3, s.double()), (4, s), (5, x), (6, -1), (6, "auto"), (6, 99), (7, w.t())):
        args = list(good)
        args[at] = bad
        assert b.gemm_rowwise(*args) is None, (at, bad)
    with pytest.raises(ValueError):
        ops.fp8_gemm_rowwise(x, w, s, s)
    with pytest.raises(NotImplementedError):
        ops.fp8_gemm_blockwise(x[:, :8], w[:, :8], s[:1].view(1, 1), s[:1].view(1, 1))


def test_without_a_device_every_call_is_left_to_the_wrappers():
    b = _lib.binding()
    x = _codes(4, 16)
    assert b.gemm_rowwise() is None and b.row_quantize(x.float()) is None and b.row_quantize("x") is None
    assert b.gemm_rowwise(x, x, x, x, None, None, 0, None, False) is None
    assert b.mark_ready(10**6) is None and b.mark_ready("cuda") is None


def _without_binding(monkeypatch, path):
    monkeypatch.setattr(_lib, "_binding", None)
    monkeypatch.setattr(_lib, "BINDING_PATH", str(path))
    with pytest.warns(RuntimeWarning, match="cannot be loaded"):
        return _lib.binding()


@pytest.mark.parametrize("content", [None, b"", b"not a shared object"])
def test_a_binding_that_cannot_be_loaded_leaves_every_call_to_the_wrappers(monkeypatch, tmp_path, content):
    path = tmp_path / "mi355x_torch_binding.so"
    if content is not None:
        path.write_bytes(content)
    b = _without_binding(monkeypatch, path)
    assert b.gemm_rowwise() is None and b.row_quantize(torch.ones(2, 2)) is None and b.mark_ready(0) is None
    assert _lib.binding() is b  # (one attempt, one warning)
    with pytest.raises(RuntimeError, match="only runs on a ROCm device"):  # (the wrappers' own check, not the loader's error)
        ops.fp8_row_quantize(torch.ones(4, 16))


@pytest.mark.gpu
def test_calls_run_without_the_binding(gpu_device, monkeypatch, tmp_path):
    calls = _calls(gpu_device)
    want = {name: _bits(call()) for name, call in calls.items()}
    _without_binding(monkeypatch, tmp_path / "missing.so")
    for name, call in calls.items():
        assert all(torch.equal(a, b) for a, b in zip(_bits(call()), want[name])), name
