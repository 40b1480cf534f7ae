"""Plans of the tiled family for rows off the 128-byte lines, which cost most configurations more: by the rows' pitch, and not on short rows."""
import pytest
import torch

from tritonbench_amd import _lib

AUTO = _lib.VARIANT_AUTO


def _planes(m, n, k):
    return _lib.load().mi355x_fp8_rowwise_workspace_bytes(m, n, k, AUTO) // (4 * m * n)


# (cut into the six or seven parts that off the lines look like a gain, these took 1.3 to 1.4 times as long)
@pytest.mark.parametrize("m,n,k", [(563, 64, 752), (293, 64, 656), (1292, 16, 704), (2735, 32, 832), (1127, 80, 832), (279, 80, 576)])
def test_short_rows_stay_whole(m, n, k):
    assert _planes(m, n, k) == _planes(m, n, -(-k // 128) * 128) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1447, 3247, 6864), (2052, 1168, 14048), (1000, 3000, 4112), (317, 825, 3312), (6603, 16, 1440), (1447, 3247, 6912)])
@pytest.mark.parametrize("side", ["on", "off"])
def test_the_plan_is_by_the_pitch(gpu_device, m, n, k, side):
    """As many parts as for rows that fill the pitch, off the lines as the query says, and the product is right."""
    lines = -(-k // 128) * 128
    ld = lines if side == "on" else k if k % 128 else k + 16
    want = _planes(m, n, lines) if side == "on" else _planes(m, n, k if k % 128 else k + 16 - 128)  # (a step's worth: off the lines, as many steps)
    print(f"case {m}x{n}x{k} pitch {ld}: {want} planes", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(m)
    a, b = (torch.randn((r, ld), generator=g, device=gpu_device).to(torch.float8_e4m3fn)[:, :k] for r in (m, n))
    sa, sb = (torch.rand(r, generator=g, device=gpu_device) + 0.5 for r in (m, n))
    space = torch.full((16, m, n), float("nan"), device=gpu_device)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    _lib.check(_lib.load().mi355x_fp8_rowwise_gemm(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), None, out.data_ptr(), m, n, k, ld, ld, n,
                                                   space.data_ptr(), 64 * m * n, AUTO, torch.cuda.current_stream().cuda_stream), "gemm")
    torch.cuda.synchronize()
    assert int(torch.isfinite(space).flatten(1).all(1).sum()) == want
    exact = (a.double() @ b.double().t()) * sa.double()[:, None] * sb.double()[None, :]
    assert ((out.double() - exact).norm() / exact.norm()).item() < 2.0**-8  # (one rounding to bf16)
