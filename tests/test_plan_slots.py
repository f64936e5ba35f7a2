"""Plans that a thread has kept are those that a search gives: more shapes than there are slots, asked for in another order, again, from
threads of their own, and for several formats in turn (which share the shape of a plan, but not its time and so not the route)."""
import itertools
import threading

import pytest

from sensenova_u1_amd import ops

SHAPES = list(itertools.product((17, 40, 64, 65, 203, 1024), (515, 4096, 12288), (256, 4096, 12288), (False, True), (0, 1 << 22, 1 << 40)))


@pytest.mark.parametrize("qt", [ops.Q8_0, ops.Q4_K, ops.Q6_K])
def test_kept_plans_are_the_searched_ones(qt):
    def ask(shapes, out):
        out.extend((s, ops.mid_plan(qt, *s)) for s in shapes if not (s[3] and s[1] % 8))

    def fresh(shapes):
        out = []
        t = threading.Thread(target=ask, args=(shapes, out))   # (a thread begins with nothing kept)
        t.start()
        t.join()
        return out

    want = {}
    for s in SHAPES:
        want.update(fresh([s]))
    assert len(set(want.values())) > 20
    assert dict(fresh(SHAPES)) == want and dict(fresh(SHAPES[::-1] + SHAPES)) == want
    again = []
    ask([s for s in SHAPES for _ in range(2)], again)
    assert dict(again) == want


@pytest.mark.parametrize("first,second", [(ops.Q4_0, ops.Q6_K), (ops.Q6_K, ops.Q4_0), (ops.Q5_K, ops.Q8_0)])
def test_kept_plans_belong_to_one_format(first, second):
    """Two formats in alternation in one thread, against a thread that has kept nothing of the other; among the shapes some whose
    route depends on the format."""
    shapes = [(m, n, k, pair, ws) for m, n, k in itertools.product((17, 24, 32, 40, 48, 64, 100, 203, 700, 1500), (512, 1024, 2056, 12288),
                                                                   (256, 2048, 4096)) for pair in (False, True) for ws in (0, 1 << 40)]
    got = {first: [], second: []}

    def alone(qt, out):
        out.extend(ops.mid_plan(qt, *s) for s in shapes)

    def together():
        for s in shapes:
            for qt in (first, second):
                got[qt].append(ops.mid_plan(qt, *s))

    want = {first: [], second: []}
    for target, args in ((alone, (first, want[first])), (alone, (second, want[second])), (together, ())):
        t = threading.Thread(target=target, args=args)
        t.start()
        t.join()
    assert sum(a != b for a, b in zip(want[first], want[second])) >= 5
    assert got == want
