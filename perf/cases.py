"""The workloads this package is timed on: FP8 linear layers as a model runs them.

A case is one linear layer `y = x @ w.T` in one of the three scalings the package offers, at one
size, with what stands in front of the product:

  scaling "row"      one scale per row of x and per row of w            ops.fp8_gemm_rowwise
  scaling "grouped"  the same per expert, rows sorted by expert         ops.fp8_gemm_rowwise_grouped
  scaling "block"    one scale per 128 x 128 block of x and of w        ops.fp8_gemm_blockwise

  front "none"       x is already e4m3fn codes and scales
  front "quantise"   x is bf16 or fp32 and is quantised in the pass
  front "rmsnorm"    x is bf16, normalised and quantised by the fused kernel
  front "silu_mul"   x is two bf16 halves of a gated MLP, gated and quantised by the fused kernel

Weights are quantised once, in prepare(), as a server does when it loads a model.
"""
import math

import torch

from tritonbench_amd import ops

SOURCE_BYTES = {"bf16": 2, "f32": 4}
SOURCE_TYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
LARGEST_FLOPS = 2 * 8192**3
LARGEST_WEIGHT = 1 << 29
LARGEST_ROWS = 1 << 29  # elements of x, and of y


def _case(m, n, k, scaling="row", front="none", source="bf16", groups=1, routed=False, bias=False, out="bf16", name=None):
    c = dict(m=m, n=n, k=k, scaling=scaling, front=front, source=source, groups=groups, routed=routed, bias=bias, out=out)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one token through a small model's projection: a few megabytes, launch-bound
        _case(1, 2304, 2048, name="row_1x2304x2048"),
        # decode with a batch of 16 against a 64 MB weight: the decode headline
        _case(16, 8192, 8192, name="row_16x8192x8192"),
        # decode with a batch of 32 through the QKV projection of a 70B model, RMSNorm in front
        _case(32, 10240, 8192, front="rmsnorm", name="rmsnorm_row_32x10240x8192"),
        # a large decode batch, or a short prompt
        _case(128, 8192, 8192, name="row_128x8192x8192"),
        # a prompt of no particular length against sizes that are no multiple of any tile, with a bias
        _case(1000, 3000, 4112, bias=True, name="row_1000x3000x4112_bias"),
        # the inner size no multiple of 16 (rows start at any byte), fp32 source, float16 result
        _case(517, 3000, 1041, front="quantise", source="f32", bias=True, out="f16", name="row_517x3000x1041_f32_f16"),
        # prefill through the down projection of a 70B model, SiLU-mul in front
        _case(1024, 8192, 28672, front="silu_mul", name="silu_row_1024x8192x28672"),
        # the square product the path is quoted on
        _case(8192, 8192, 8192, name="row_8192x8192x8192"),
        # mixture of experts: prefill in equal groups, and a routed decode batch quantised in the pass
        _case(8192, 4096, 4096, scaling="grouped", groups=4, name="grouped_4_8192x4096x4096"),
        _case(128, 4096, 4096, scaling="grouped", groups=16, routed=True, front="quantise", name="grouped_16_128x4096x4096"),
        # block scaling: decode and prefill, the activation quantised in the pass
        _case(16, 8192, 8192, scaling="block", front="quantise", name="block_16x8192x8192"),
        _case(4096, 8192, 8192, scaling="block", front="quantise", name="block_4096x8192x8192"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        scaling = rng.choices(("row", "grouped", "block"), (5, 2, 3))[0]
        m = _log_int(rng, 1, 16384)
        n = _log_int(rng, 512, 57344)
        k = _log_int(rng, 512, 28672)
        # widths of models are multiples of 64 to 512 as a rule; the others are taken as they come
        step = rng.choice((512, 256, 128, 64, 16))
        if rng.random() < 0.75:
            n = max(step, n // step * step)
        groups, routed, bias, out, front, source = 1, False, False, "bf16", "none", "bf16"
        # only the row-wise product takes rows that start at any byte
        odd = scaling == "row" and rng.random() < 0.2
        if not odd:
            k = max(512, k // step * step)
        if scaling == "grouped":
            groups = _log_int(rng, 2, 64)
            routed = rng.random() < 0.7
            if not routed:
                m = max(1, m // groups) * groups
        elif scaling == "row":
            bias = rng.random() < 0.3
            out = "f16" if rng.random() < 0.2 else "bf16"
        fronts = ("none", "quantise") if odd or scaling == "block" else ("none", "quantise", "rmsnorm", "silu_mul")
        front = rng.choice(fronts)
        if front == "quantise" and rng.random() < 0.25:
            source = "f32"
        if 2 * m * n * k <= LARGEST_FLOPS // (16 if odd else 1) and groups * n * k <= LARGEST_WEIGHT and m * max(n, k) <= LARGEST_ROWS:
            return _case(m, n, k, scaling, front, source, groups, routed, bias, out)


def _sizes(case, g):
    """Rows of each expert: equal, or every row sent to an expert at random."""
    m, groups = case["m"], case["groups"]
    if not case["routed"]:
        return torch.full((groups,), m // groups, dtype=torch.int32, device="cuda")
    to = torch.randint(0, groups, (m,), generator=g, device="cuda")
    return torch.bincount(to, minlength=groups).to(torch.int32)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    m, n, k = case["m"], case["n"], case["k"]
    quantise = ops.fp8_block_quantize if case["scaling"] == "block" else ops.fp8_row_quantize

    def normal(*shape, scale=1.0, dtype=torch.bfloat16):
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(scale)

    s = {"case": case}
    s["w"], s["w_scale"] = quantise(normal(case["groups"] * n, k, scale=0.02))
    s["bias"] = normal(n, scale=0.1) if case["bias"] else None
    s["out_dtype"] = torch.float16 if case["out"] == "f16" else torch.bfloat16
    x = normal(m, k, dtype=SOURCE_TYPES[case["source"]])
    if case["front"] == "none":
        s["x"], s["x_scale"] = quantise(x)
        # what a program that calls the product again and again keeps: its result and its workspace
        s["out"] = torch.zeros((m, n), dtype=s["out_dtype"], device="cuda")
        s["workspace"] = ops.gemm_workspace(m, n, k, x.device) if case["scaling"] == "row" else None
    else:
        s["x"] = x
        s["out"] = s["workspace"] = None
        if case["front"] == "rmsnorm":
            s["norm_weight"] = normal(k, scale=0.1).add_(1.0)
        elif case["front"] == "silu_mul":
            s["x2"] = normal(m, k)
    if case["scaling"] == "grouped":
        s["m_sizes"] = _sizes(case, g)
    return s


def run(state):
    case = state["case"]
    front = case["front"]
    if front == "none":
        xq, x_scale = state["x"], state["x_scale"]
    elif front == "rmsnorm":
        xq, x_scale = ops.rms_norm_fp8_rowwise_quant(state["x"], state["norm_weight"])
    elif front == "silu_mul":
        xq, x_scale = ops.silu_mul_fp8_rowwise_quant(state["x"], state["x2"])
    elif case["scaling"] == "block":
        xq, x_scale = ops.fp8_block_quantize(state["x"])
    else:
        xq, x_scale = ops.fp8_row_quantize(state["x"])
    if case["scaling"] == "grouped":
        return ops.fp8_gemm_rowwise_grouped(xq, state["w"], state["m_sizes"], x_scale, state["w_scale"], out=state["out"])
    if case["scaling"] == "block":
        return ops.fp8_gemm_blockwise(xq, state["w"], x_scale, state["w_scale"], out=state["out"])
    return ops.fp8_gemm_rowwise(xq, state["w"], x_scale, state["w_scale"], bias=state["bias"], out=state["out"],
                                workspace=state["workspace"], out_dtype=state["out_dtype"])


def work(case):
    m, n, k, groups = case["m"], case["n"], case["k"], case["groups"]
    # experts that get a row at all: the others' weights need not be read
    used = groups * (1 - (1 - 1 / groups) ** m) if case["routed"] else groups
    if case["scaling"] == "block":
        x_scales, w_scales = -(-m // 128) * -(-k // 128), -(-n // 128) * -(-k // 128)
    else:
        x_scales, w_scales = m, used * n
    nbytes = used * n * k + 4 * w_scales + 2 * m * n + (2 * n if case["bias"] else 0)
    if case["front"] == "none":
        nbytes += m * k + 4 * x_scales
    else:
        nbytes += m * k * SOURCE_BYTES[case["source"]] * (2 if case["front"] == "silu_mul" else 1)
        nbytes += 2 * k if case["front"] == "rmsnorm" else 0
    return {"bytes": nbytes, "flops": 2 * m * n * k}


def tolerance(case):
    # Four times the distance from the same codes and scales multiplied out in float64, measured over the
    # listed cases: 1.66e-3 (largest single value 3.9e-3) for a bfloat16 result, 2.1e-4 (4.9e-4) for a
    # float16 one, nearly all of it the one rounding of the result. The fused front ends' own results differ from
    # float64 ones by a code in 1e4 (ties): 1.9e-3 (1.2e-2).
    if case["front"] in ("rmsnorm", "silu_mul"):
        return {"rel": 7.6e-3, "max": 4.8e-2} if case["out"] == "bf16" else {"rel": 3.7e-3, "max": 4.8e-2}
    return {"rel": 6.6e-3, "max": 1.6e-2} if case["out"] == "bf16" else {"rel": 8.4e-4, "max": 2e-3}
