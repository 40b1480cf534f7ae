"""The choice for a shape is a function of its sizes: the table of the latest shapes a thread keeps changes no answer."""
import random
import threading

import pytest
import torch

from tritonbench_amd import _lib


def _answers(shapes):
    lib = _lib.load()
    return [
        (lib.mi355x_fp8_rowwise_select_variant(m, n, k), lib.mi355x_fp8_rowwise_workspace_bytes(m, n, k, v))
        for m, n, k in shapes
        for v in (_lib.VARIANT_AUTO, _lib.VARIANT_TILED, _lib.VARIANT_TILED | 2 << 8, _lib.VARIANT_TILED | 3 << 16)
    ]


def test_answers_do_not_depend_on_the_calls_before():
    rng = random.Random(5)
    # (more shapes than the table has entries, among them ones that differ in one size only)
    shapes = [(rng.choice((1, 2, 16, 64, 100, 1000)), rng.choice((512, 2304, 8192)) + 16 * rng.randrange(4), 16 * rng.randrange(32, 1800))
              for _ in range(700)]
    first = _answers(shapes)
    order = list(range(len(shapes)))
    rng.shuffle(order)
    again = [None] * len(first)
    for i in order:
        again[4 * i:4 * i + 4] = _answers(shapes[i:i + 1])
    assert again == first
    assert [_answers([s])[0] for s in shapes for _ in range(2)][::2] == first[::4]

    results = [None] * 4  # (a thread of its own starts with an empty table)

    def work(t):
        part = shapes[t::4]
        results[t] = _answers(part) == [a for i in range(t, len(shapes), 4) for a in first[4 * i:4 * i + 4]]

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert results == [True] * 4


def _in_a_thread_of_its_own(question):
    """The answer of an empty table."""
    answer = []
    t = threading.Thread(target=lambda: answer.append(question()))
    t.start()
    t.join()
    return answer[0]


def test_block_plans_do_not_depend_on_the_calls_before():
    lib = _lib.load()
    rng = random.Random(7)
    shapes = [(rng.choice((1, 16, 40, 64, 100, 300, 1000)), rng.choice((512, 1000, 2304)) + 16 * rng.randrange(4), 16 * rng.randrange(32, 1800))
              for _ in range(300)]
    alone = [_in_a_thread_of_its_own(lambda: lib.mi355x_fp8_blockwise_workspace_bytes(*s)) for s in shapes]
    assert 50 < sum(a > 0 for a in alone) < 250
    for _ in range(3):
        order = list(range(len(shapes)))
        rng.shuffle(order)
        for i in order:
            assert lib.mi355x_fp8_blockwise_workspace_bytes(*shapes[i]) == alone[i], shapes[i]


def test_each_plan_of_a_shape_is_known_by_itself():
    """Each pinned plan against its answer alone, in any order: what else a shape was asked for changes nothing."""
    lib = _lib.load()
    rng = random.Random(11)
    shapes = [(rng.choice((16, 64, 100, 300)), 512 + 16 * rng.randrange(64), 4096 + 16 * rng.randrange(512)) for _ in range(40)]
    variants = [_lib.VARIANT_AUTO, *(_lib.tiled_variant(c, s) for c in (None, 0, 3) for s in (0, 2, 3, 5))]
    pairs = [(s, v) for s in shapes for v in variants]
    alone = {p: _in_a_thread_of_its_own(lambda: lib.mi355x_fp8_rowwise_workspace_bytes(*p[0], p[1])) for p in pairs}
    for (m, n, k), v in pairs:  # (whole rounds of a pinned factor are the plan's own: 33 and more steps hold 2, 3 and 5 parts)
        if v >> 16:
            assert alone[(m, n, k), v] == (v >> 16) * 4 * m * n
    assert len({alone[s, v] // (4 * s[0] * s[1]) for s, v in pairs}) >= 5
    for _ in range(3):
        rng.shuffle(pairs)
        for s, v in pairs:
            assert lib.mi355x_fp8_rowwise_workspace_bytes(*s, v) == alone[s, v], (s, v)


@pytest.mark.gpu
def test_full_and_short_workspaces_take_turns(gpu_device):
    """A call with a short workspace runs the plan that fits it, whichever plan the shape ran before."""
    m, n, k = 264, 640, 8192
    lib = _lib.load()
    g = torch.Generator(device=gpu_device).manual_seed(3)
    codes = lambda r: torch.randn((r, k), generator=g, device=gpu_device).to(torch.float8_e4m3fn)
    xq, wq = codes(m), codes(n)
    xs, ws = (torch.rand(r, generator=g, device=gpu_device) + 0.5 for r in (m, n))
    need = lib.mi355x_fp8_rowwise_workspace_bytes(m, n, k, _lib.VARIANT_AUTO)
    planes = need // (4 * m * n)
    assert planes >= 3
    stream = torch.cuda.current_stream().cuda_stream

    def run(parts):
        """The result, and how many planes of partial sums the call left behind."""
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
        space = torch.full((planes, m, n), float("nan"), device=gpu_device)
        print(f"case {m}x{n}x{k} {parts} planes", flush=True)
        _lib.check(lib.mi355x_fp8_rowwise_gemm(xq.data_ptr(), wq.data_ptr(), xs.data_ptr(), ws.data_ptr(), None, out.data_ptr(), m, n, k, k, k, n,
                                               space.data_ptr(), parts * 4 * m * n, _lib.VARIANT_AUTO, stream), "gemm")
        torch.cuda.synchronize()
        written = torch.isfinite(space).flatten(1)
        assert torch.equal(written.any(1), written.all(1))
        return out.view(torch.int16).cpu(), int(written.all(1).sum())

    alone = {parts: _in_a_thread_of_its_own(lambda: run(parts)) for parts in (planes, 2, 0)}
    assert alone[planes][1] == planes and alone[2][1] <= 2 and alone[0][1] == 0
    exact = (xq.double() @ wq.double().t()) * xs.double()[:, None] * ws.double()[None, :]
    for parts in (planes, 2, 0, planes, 0, 2, planes):
        got, written = run(parts)
        assert torch.equal(got, alone[parts][0]) and written == alone[parts][1]
        result = got.view(torch.bfloat16).to(gpu_device).double()
        assert ((result - exact).norm() / exact.norm()).item() < 2.0**-8  # (one rounding to bf16)
