"""The choice for a shape is a function of its sizes: the table of the latest shapes a thread keeps changes no answer."""
import random
import threading

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
