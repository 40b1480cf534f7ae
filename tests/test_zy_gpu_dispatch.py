"""The automatic choice of kernel family, tile configuration and split factor against the pinned
alternatives, timed on the device: the cost estimates behind the choice are tables of measured
constants, and a table that has drifted away from the kernels shows here as a choice that is
clearly slower than one of its alternatives. Needs an MI355X.

Timing (tritonbench_amd/tuning.py, the module behind the autotuned backend): a captured graph of
16 launches over rotating operand sets (cold weights, as a model's are), sustained bursts, the
median of three. The bar is 25 %: repeated measurements of one and the same plan on the shorter of
these shapes (10-30 us) differ by up to 8 % within a run (1 x 8192 x 16384 and 2048^3 have both shown
the automatic choice and the identical pinned plan that far apart), and plans of two launches move
more than that from run to run: 1024 x 1024 x 8192 in four splits has measured 19.7 to 26.8 us over
eight runs (its second kernel alone 4.9 to 7.1) with the unsplit plans beside it steady to 0.1 us.
A table that has drifted shows well beyond the bar (the 128x256 constants once put nineteen small
shapes 30-45 % off).

These are wall-clock assertions, not parity: they carry the `perf` marker beside `gpu`
(`-m "gpu and not perf"` leaves them out), every shape prints its margin, and the file sorts behind
every parity file so that a noisy replay cannot keep `pytest -x` from reaching those."""
import pytest
import torch

from tritonbench_amd import _lib, tuning

pytestmark = [pytest.mark.gpu, pytest.mark.perf]

TOLERANCE = 1.25
# decode- and small-prefill-sized rows of the Llama-3-70B projection sweep, and the small ragged shape with bias
SHAPES = [(32, 8192, 8192, False), (64, 8192, 8192, False), (128, 8192, 8192, False), (128, 10240, 8192, False),
          (32, 10240, 8192, False), (256, 8192, 8192, False), (1000, 3000, 4112, True),
          (128, 8192, 4096, False), (128, 8192, 28672, False), (256, 4096, 8192, False),
          (64, 4096, 8192, False), (128, 2048, 8192, False),
          # the rest of the decode rows (M = 1, 32, 128) of the Llama-3-70B sweep
          (1, 8192, 8192, False), (1, 10240, 8192, False), (1, 57344, 8192, False), (1, 8192, 28672, False),
          (32, 57344, 8192, False), (32, 8192, 28672, False), (128, 57344, 8192, False),
          # one tile row of 256x256 tiles with streamed B; several tile rows of the smaller configurations
          (256, 57344, 8192, False), (512, 16384, 16384, False),
          # decode-sized rows of the reference operator's own default sweep (operator.py:107-128); the
          # first is the shape of its stored run configuration
          (16, 13312, 13312, False), (1, 8192, 16384, False), (4, 13312, 2048, False), (8, 8192, 6656, False),
          (16, 4096, 6656, False), (32, 2304, 16384, False), (32, 8192, 13312, False), (64, 13312, 2048, False),
          (128, 2304, 6656, False), (128, 8192, 2304, False),
          # at most one 128x128 work item per CU: the deep-ring configuration, unsplit and split
          (1024, 2048, 4096, False), (2048, 2048, 2048, False), (1024, 1024, 8192, False), (1024, 2048, 16384, False),
          (768, 2048, 2048, False),
          # narrow panels with long rows: a few workgroups that each stream a long tile
          (1, 2048, 28672, False), (8, 1024, 28672, False), (16, 1024, 16384, False),
          # a vocabulary-wide panel with short rows (the output projection of a small model)
          (1, 128256, 2048, False), (8, 128256, 2048, False), (1, 151936, 1536, False)]


@pytest.mark.parametrize("m,n,k,bias", SHAPES)
def test_automatic_choice_is_close_to_the_best_alternative(gpu_device, m, n, k, bias):
    print(f"case m={m} n={n} k={k} bias={bias}", flush=True)
    dev = gpu_device
    # operand sets to rotate through: more than twice the 256 MB memory-side cache in total, as the
    # cost tables are calibrated on operands that come from HBM
    sets = tuning.make_operand_sets(m, n, k, bias, dev)
    alternatives = tuning.candidates(m, n, k)
    # two rounds over all candidates, the automatic choice first and last: whatever is timed first
    # runs on a colder clock
    # (further rounds, up to five in all, only if the bound does not hold after two: one noisy replay must not
    # fail the suite; every timing call runs on a fresh stream, so the rounds also see different hardware queues)
    times, auto = {name: float("inf") for name in alternatives}, float("inf")
    for rnd in range(5):
        auto = min(auto, tuning.time_variant_us(sets, _lib.VARIANT_AUTO))
        for name, v in alternatives.items():
            times[name] = min(times[name], tuning.time_variant_us(sets, v))
        auto = min(auto, tuning.time_variant_us(sets, _lib.VARIANT_AUTO))
        if rnd >= 1 and auto <= TOLERANCE * min(times.values()):
            break
    best_name = min(times, key=times.get)
    print(f"  automatic {auto:.1f} us = {auto / times[best_name]:.3f} x best ('{best_name}' {times[best_name]:.1f} us; "
          f"bar {TOLERANCE:.2f}); " + ", ".join(f"{nm} {t:.1f}" for nm, t in times.items()), flush=True)
    assert auto <= TOLERANCE * times[best_name], (
        f"automatic choice takes {auto:.1f} us, '{best_name}' {times[best_name]:.1f} us: the cost tables need recalibrating")


def _time_us(call, sets, burst_us=4000.0):
    """Microseconds per call(i) over operand sets i: a captured graph of 16, the median of three bursts, on a stream of its own."""
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call(0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for i in range(16):
                call(i % sets)

        def burst(replays):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record(stream)
            for _ in range(replays):
                graph.replay()
            end.record(stream)
            stream.synchronize()
            return start.elapsed_time(end) * 1e3 / (16 * replays)

        burst(1)
        replays = max(1, int(burst_us / (16 * max(burst(1), 1.0))))
        return sorted(burst(replays) for _ in range(3))[1]


# the generic family's tiles, which no argument pins: a product with fewer columns or a shorter K takes no longer than the one with
# more, within 5 % (with lines drawn by tile counts and K 1358x23320x1817 took 199 us and 179 with K = 2051)
@pytest.mark.parametrize("less,more", [((1024, 8064, 3145), (1024, 8192, 3145)), ((1358, 23320, 1817), (1358, 23320, 2051))])
def test_generic_tiles_follow_the_work(gpu_device, less, more):
    times = {}
    for m, n, k in (less, more):
        print(f"case {m}x{n}x{k}", flush=True)
        sets = tuning.make_operand_sets(m, n, k, False, gpu_device)
        times[m, n, k] = min(tuning.time_variant_us(sets, _lib.VARIANT_GENERIC) for _ in range(3))
    print("  " + ", ".join(f"{s}: {t:.1f} us" for s, t in times.items()), flush=True)
    assert times[less] <= 1.05 * times[more]


# the block-scaled forms: decode and prefill sizes, and wide panels with short rows or rows off the 128-byte lines, where the
# streaming forms are behind the plain 128x128 tiles
@pytest.mark.parametrize("m,n,k", [(1, 2304, 2048), (16, 8192, 8192), (32, 8192, 8192), (64, 57344, 8192), (128, 8192, 8192),
                                   (512, 4096, 4096), (4096, 4096, 4096), (44, 87564, 32), (49, 18200, 64), (128, 100096, 256),
                                   (128, 40064, 512), (64, 65536, 128), (9, 64149, 3952), (16, 58376, 4112), (1, 58376, 6688),
                                   (2, 63172, 4128), (1, 24904, 1424), (64, 19696, 11024)])
def test_block_scaled_choice_is_close_to_the_best_form(gpu_device, m, n, k):
    lib = _lib.load()
    g = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    codes = lambda r: torch.randn((r, k), generator=g, device=gpu_device, dtype=torch.bfloat16).to(torch.float8_e4m3fn)
    factors = lambda r: torch.rand((-(-r // 128), -(-k // 128)), generator=g, device=gpu_device) + 0.5
    count = min(8, max(2, 600_000_000 // (n * k)))
    sets = [(codes(m), codes(n), factors(m), factors(n), torch.empty((m, n), dtype=torch.bfloat16, device=gpu_device)) for _ in range(count)]

    def call(form):
        def one(i):
            x, w, xs, ws, out = sets[i]
            _lib.check(lib.mi355x_fp8_blockwise_gemm_ex(x.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), out.data_ptr(), m, n, k,
                                                        k, k, n, form, torch.cuda.current_stream().cuda_stream), "blockwise_gemm_ex")
        return one
    forms = [f for f in range(5) if (f != _lib.BLOCK_ONE_TILE or m <= 64) and (f != _lib.BLOCK_NARROW or _lib.skinny_family_takes(m, n))]
    times, auto = {f: float("inf") for f in forms}, float("inf")
    for rnd in range(4):
        auto = min(auto, _time_us(call(-1), count))
        for f in forms:
            times[f] = min(times[f], _time_us(call(f), count))
        if auto <= TOLERANCE * min(times.values()):
            break
    print(f"  {m}x{n}x{k}: form {lib.mi355x_fp8_blockwise_form(m, n, k)} {auto:.1f} us; " +
          ", ".join(f"{f}: {t:.1f}" for f, t in times.items()), flush=True)
    assert auto <= TOLERANCE * min(times.values())


# the grouped forms against the pinned tile configurations, rows sent to groups at random or half of them to one group, rows of B on
# and off the 128-byte lines
@pytest.mark.parametrize("g,m,n,k,hot", [(16, 128, 4096, 4096, False), (16, 128, 4096, 4112, False), (8, 64, 14336, 4112, False),
                                         (64, 512, 4096, 4096, True), (16, 512, 4096, 4096, True), (8, 256, 14336, 4096, True),
                                         (16, 400, 4096, 2064, False), (8, 700, 4096, 4112, False), (12, 1200, 6000, 6672, False),
                                         (16, 939, 1792, 4736, True), (32, 1800, 4096, 4096, True), (4, 8192, 4096, 4096, False)])
def test_grouped_choice_is_close_to_the_best_tiles(gpu_device, g, m, n, k, hot):
    lib = _lib.load()
    gen = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    codes = lambda r: torch.randn((r, k), generator=gen, device=gpu_device, dtype=torch.bfloat16).to(torch.float8_e4m3fn)
    count = min(6, max(2, 600_000_000 // (g * n * k)))
    to = torch.randint(0, g, (m,), generator=gen, device=gpu_device)
    if hot:
        to[: m // 2] = g // 2
    sizes = torch.bincount(to, minlength=g).to(torch.int32)
    xs, ws = torch.rand(m, generator=gen, device=gpu_device), torch.rand(g * n, generator=gen, device=gpu_device)
    sets = [(codes(m), codes(g * n), torch.empty((m, n), dtype=torch.bfloat16, device=gpu_device)) for _ in range(count)]

    def call(config):
        def one(i):
            x, w, out = sets[i]
            _lib.check(lib.mi355x_fp8_rowwise_grouped_gemm(x.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), sizes.data_ptr(),
                                                           out.data_ptr(), g, m, n, k, k, k, n, config,
                                                           torch.cuda.current_stream().cuda_stream), "grouped_gemm")
        return one
    times, auto = {c: float("inf") for c in range(_lib.NUM_GROUPED_TILE_CONFIGS)}, float("inf")
    for rnd in range(4):
        auto = min(auto, _time_us(call(-1), count))
        for c in times:
            times[c] = min(times[c], _time_us(call(c), count))
        if auto <= TOLERANCE * min(times.values()):
            break
    print(f"  {g} groups {m}x{n}x{k} hot={hot}: form {lib.mi355x_fp8_rowwise_grouped_form(g, m, n, k)} {auto:.1f} us; " +
          ", ".join(f"{c}: {t:.1f}" for c, t in times.items()), flush=True)
    assert auto <= TOLERANCE * min(times.values())
