"""The grouped GEMM's forms for few rows a group, at the sizes where they can go wrong, against the pinned 128x128 tiles
(which the oracle checks). Integer codes and power-of-two scales: every sum is below 2^24 and exact in f32 whatever its
order, so the results have to agree bit for bit. Needs an MI355X."""
import pytest
import torch

from tritonbench_amd import _lib, ops

pytestmark = pytest.mark.gpu

SMALL_TILES = 1  # tile configuration 128x128


def _operands(dev, g, m, n, k, seed=0):
    gen = torch.Generator().manual_seed(seed)
    ints = lambda *s: torch.randint(-4, 5, s, generator=gen).to(torch.float32).to(torch.float8_e4m3fn)
    powers = lambda s: 2.0 ** torch.randint(-3, 4, (s,), generator=gen).to(torch.float32)
    return ints(m, k).to(dev), ints(g * n, k).to(dev), powers(m).to(dev), powers(g * n).to(dev)


def _spread(g, m, seed=0):
    to = torch.randint(0, g, (m,), generator=torch.Generator().manual_seed(seed))
    return torch.bincount(to, minlength=g).tolist()


CASES = [
    # g, m, n, k, sizes (None: rows sent to groups at random)
    # up to 8 rows a group on average
    (1, 1, 16, 16, [1]),
    (2, 16, 33, 144, [16, 0]),               # one whole block, N one past a tile, K tail
    (2, 16, 31, 1024, [0, 16]),
    (4, 31, 130, 272, [17, 0, 13, 1]),       # a group of two blocks
    (16, 128, 512, 1040, None),
    (64, 300, 64, 2048, None),
    (65, 200, 40, 128, None),                # more groups than lanes: two rounds of the look-up
    (130, 900, 96, 256, None),               # three rounds, tiles not a multiple of the XCDs
    (256, 256, 32, 128, None),
    (200, 64, 32, 128, [0] * 199 + [64]),    # the last group holds everything
    (8, 60, 128, 512, [-3, 20, 2**31 - 1, 5, 0, 7, 1, 2]),  # sizes that lie: cut off at M
    (8, 64, 128, 512, [3, 0, 9, 5, 0, 7, 1, 2]),            # rows past the sum stay untouched
    # few tiles, long rows: 32- and 64-row blocks
    (2, 32, 128, 4096, [31, 1]),
    (2, 32, 72, 4112, [0, 32]),
    (3, 49, 130, 4096, [33, 0, 16]),
    (2, 64, 128, 4096, [64, 0]),
    (2, 63, 40, 4240, [5, 58]),
    (2, 50, 128, 4096, [2**31 - 1, 2**31 - 1]),
    # tiles with the streaming policy
    (16, 200, 1024, 2048, None),
    (16, 1024, 1000, 2064, None),
    (8, 500, 2048, 2048, [129, 0, 127, 128, 1, 0, 100, 5]),
    (16, 1100, 2048, 2064, None),            # 65 to 128 rows a group: 128x256 tiles
    (16, 2048, 2040, 2048, [128] * 16),
    (16, 1500, 2048, 2048, [1000] + [0] * 14 + [400]),
]


# the form each of these runs, so that the cases above keep reaching what they are there for
@pytest.mark.parametrize("form,shapes", [
    (_lib.GROUPED_ROWS_16, [(1, 1, 16, 16), (2, 16, 33, 144), (16, 128, 512, 1040), (65, 200, 40, 128), (256, 256, 32, 128), (8, 64, 128, 512)]),
    (_lib.GROUPED_ROWS_32, [(2, 32, 128, 4096), (2, 32, 72, 4112)]),
    (_lib.GROUPED_ROWS_64, [(3, 49, 130, 4096), (2, 64, 128, 4096), (2, 63, 40, 4240)]),
    (_lib.GROUPED_STREAM_128, [(16, 200, 1024, 2048), (8, 500, 2048, 2048), (16, 700, 1000, 2048)]),
    (_lib.GROUPED_STREAM_256, [(16, 2048, 2040, 2048), (16, 1500, 2048, 2048), (4, 480, 11584, 9536)]),
    (_lib.GROUPED_TILES, [(16, 1024, 1000, 2064), (16, 1100, 2048, 2064), (8, 700, 4096, 4112), (4, 8192, 4096, 4096)]),
])
def test_the_cases_reach_the_forms(form, shapes):
    for shape in shapes:
        assert _lib.load().mi355x_fp8_rowwise_grouped_form(*shape) == form, shape


# rows of K bytes in rows of a longer pitch: a partial last step of rows on the 128-byte lines (the streaming tiles with a K tail),
# and whole steps of rows off them; groups of no, one, two and more tile rows side by side
@pytest.mark.parametrize("g,m,n,k,pitch", [(16, 700, 1000, 2064, 2176), (16, 1500, 2048, 2064, 2176), (16, 100, 96, 640, 656),
                                           (16, 700, 1000, 2048, 2064), (4, 450, 11264, 2048, 2064), (2, 64, 128, 4096, 4112)])
def test_pitches_on_and_off_the_lines(gpu_device, g, m, n, k, pitch):
    x, w, xs, ws = _operands(gpu_device, g, m, n, k)
    wide = torch.full((g * n, pitch), 0x7F, dtype=torch.uint8, device=gpu_device).view(torch.float8_e4m3fn)  # (NaN beside the rows)
    wide[:, :k].copy_(w)
    sizes = _spread(g, m)
    hot = max(range(g), key=lambda i: sizes[i])
    for i in range(g):  # a group of several tile rows, and some of none
        if i != hot and i % 3 == 0:
            sizes[hot] += sizes[i]
            sizes[i] = 0
    ms = torch.tensor(sizes, dtype=torch.int32, device=gpu_device)
    got = ops.fp8_gemm_rowwise_grouped(x, wide[:, :k], ms, xs, ws)
    assert torch.equal(got, ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, tile_config=SMALL_TILES))


@pytest.mark.parametrize("g,m,n,k,sizes", CASES)
def test_forms_equal_the_small_tiles_bit_for_bit(gpu_device, g, m, n, k, sizes):
    x, w, xs, ws = _operands(gpu_device, g, m, n, k)
    ms = torch.tensor(sizes if sizes is not None else _spread(g, m), dtype=torch.int32, device=gpu_device)
    outs = []
    for cfg in (-1, SMALL_TILES):
        out = torch.full((m, n + 3), 7.0, dtype=torch.bfloat16, device=gpu_device)  # (a pitch that is no multiple of 4)
        ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, out=out[:, :n], tile_config=cfg)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])
    owned = min(m, sum(max(v, 0) for v in ms.tolist()))
    assert torch.all(outs[0][owned:] == 7.0) and torch.all(outs[0][:, n:] == 7.0)


def test_a_captured_launch_follows_new_sizes(gpu_device):
    g, m, n, k = 16, 100, 96, 640
    x, w, xs, ws = _operands(gpu_device, g, m, n, k)
    ms = torch.tensor(_spread(g, m), dtype=torch.int32, device=gpu_device)
    out = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
    call = lambda: ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, out=out)
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seed in range(3):
        ms.copy_(torch.tensor(_spread(g, m, seed + 5), dtype=torch.int32))
        want = ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, tile_config=SMALL_TILES)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


# (a form of each kernel; N a whole number of 16-byte pieces or not; no rest, a row, nearly everything, everything)
@pytest.mark.parametrize("g,m,n,k", [(16, 100, 96, 640), (16, 100, 97, 640), (2, 32, 128, 4096), (8, 500, 2048, 2048), (16, 1100, 2048, 2048),
                                     (3, 900, 520, 256), (3, 900, 513, 256), (4, 4096, 4096, 512), (130, 900, 64, 256)])
@pytest.mark.parametrize("rest", ["none", "a row", "most", "all"])
def test_a_result_made_by_the_call_is_zero_past_the_groups(gpu_device, g, m, n, k, rest):
    x, w, xs, ws = _operands(gpu_device, g, m, n, k)
    rows = {"none": m, "a row": m - 1, "most": 3, "all": 0}[rest]
    ms = torch.tensor(_spread(g, rows), dtype=torch.int32, device=gpu_device)
    want = torch.zeros((m, n), dtype=torch.bfloat16, device=gpu_device)
    ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, out=want)
    for config in (-1, 0, 1, 2):
        # (through the C entry, on memory known to hold NaN; a result that the wrapper makes may lie in memory that is zero by luck)
        got = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
        st = _lib.load().mi355x_fp8_rowwise_grouped_gemm_ex(
            x.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), ms.data_ptr(), got.data_ptr(), g, m, n, k,
            x.stride(0), w.stride(0), got.stride(0), config, 1, torch.cuda.current_stream().cuda_stream)
        _lib.check(st, "mi355x_fp8_rowwise_grouped_gemm_ex")
        assert torch.equal(got, want), config
        assert torch.equal(ops.fp8_gemm_rowwise_grouped(x, w, ms, xs, ws, tile_config=config), want), config


def test_columns_beyond_the_16_row_forms_grid(gpu_device):
    g, m, n, k = 256, 256, 2200000, 16  # (a column tile of 32 and a row block of 16 are 256 lanes, 2^32 a launch)
    x = torch.ones((m, k), device=gpu_device).to(torch.float8_e4m3fn)
    w = torch.full((g * n * k,), 0x38, dtype=torch.uint8, device=gpu_device).view(torch.float8_e4m3fn).view(g * n, k)
    scale = torch.arange(g, device=gpu_device, dtype=torch.float32).add_(1)
    ms = torch.ones(g, dtype=torch.int32, device=gpu_device)
    got = ops.fp8_gemm_rowwise_grouped(x, w, ms, torch.ones(m, device=gpu_device), scale.repeat_interleave(n))
    torch.cuda.synchronize()
    assert torch.equal(got, (scale * k).to(torch.bfloat16)[:, None].expand(m, n))
