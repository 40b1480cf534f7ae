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


# (cut into more parts on the lines than off them)
@pytest.mark.parametrize("m,n,k", [(10605, 243, 10720), (1196, 205, 11840), (522, 3880, 10208), (265, 9949, 17568), (6219, 248, 12656), (515, 818, 2256),
                                   (303, 142, 9328), (1568, 2132, 19312), (4805, 553, 23088), (283, 3747, 26224), (8276, 300, 21536)])
def test_the_query_is_enough_for_padded_rows(m, n, k):
    """The query knows of no pitch: it names as many planes as rows want that are padded onto the lines."""
    assert _planes(m, n, k) >= _planes(m, n, -(-k // 128) * 128) > 0


@pytest.mark.gpu
def test_the_plan_is_by_the_pitch(gpu_device):
    """With the workspace that the query names: rows that are or are padded onto the lines in as many parts as rows that fill the pitch, and
    the product is right on either pitch."""
    parts = []
    for m, n, k in ((1447, 3247, 6864), (2052, 1168, 14048), (522, 3880, 10208), (317, 825, 3312), (1000, 3000, 4112), (6603, 16, 1440), (1447, 3247, 6912)):
        g = torch.Generator(device=gpu_device).manual_seed(m)
        on = -(-k // 128) * 128
        need = 4 * m * n * _planes(m, n, k)
        written = []
        for ld in (on, k if k % 128 else k + 16):
            print(f"case {m}x{n}x{k} pitch {ld}", flush=True)
            a, b = (torch.randn((r, ld), generator=g, device=gpu_device).to(torch.float8_e4m3fn)[:, :k] for r in (m, n))
            sa, sb = (torch.rand(r, generator=g, device=gpu_device) + 0.5 for r in (m, n))
            space = torch.full((16, m, n), float("nan"), device=gpu_device)
            out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
            _lib.check(_lib.load().mi355x_fp8_rowwise_gemm(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), None, out.data_ptr(), m, n, k,
                                                           ld, ld, n, space.data_ptr(), need if k % 128 else space.nbytes, AUTO,
                                                           torch.cuda.current_stream().cuda_stream), "gemm")
            torch.cuda.synchronize()
            written.append(int(torch.isfinite(space).flatten(1).all(1).sum()))
            exact = (a.double() @ b.double().t()) * sa.double()[:, None] * sb.double()[None, :]
            assert ((out.double() - exact).norm() / exact.norm()).item() < 2.0**-8  # (one rounding to bf16)
        assert written[0] == _planes(m, n, on)
        parts.append(written)
    assert any(w[0] != w[1] for w in parts)  # (else nothing above told the two pitches apart)
