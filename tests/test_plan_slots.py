"""Plans that a thread has kept are those that a search gives: more shapes than there are slots, asked for in another order, again, and
from threads of their own."""
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
