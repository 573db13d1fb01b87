"""GPU test of the mixed walk's groups of far-apart heavy bodies, whose boxes
cover the system: their stacks fill up, so fewer ranges are popped at once
(the training walk of the learned form pops one at a time instead), and a
block shares them once their work is known.  A walk by lone wavefronts and the
shared one give the same bits; the two pop rules visit the same nodes and list
the same entries, in another order."""
import sys

import numpy as np
import pytest

from test_gpu_walk_share import DT, walk

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n,seed", [(30000, 20), (30000, 31), (60000, 20)])
def test_wide_group(bh, n, seed):
    say("wide group", n, seed)
    data = bh.generate(bh.GEN_BELT, seed, n)
    lone = walk(bh, data, 1.05, 64, bh.SCHED_KEY_ORDER, 1)
    shared = walk(bh, data, 1.05, 64, bh.SCHED_KEY_ORDER, 0)
    for a, b in zip(lone, shared):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    first, visit = lone[0][2], lone[0][4]
    g = int(visit.argmax())
    assert visit[g] > 5 * np.median(visit)   # the case holds such a group

    def first_step(form):
        with bh.Engine(form=form, theta=1.05) as e:
            e.set_bodies(*data)
            e.step(1, DT)
            return e.get_bodies(), e.groups()

    (sa, ga), (sb, gb) = first_step(bh.FORM_MIXED), first_step(bh.FORM_LEARNED)
    assert np.array_equal(sa["ids"], sb["ids"]) and np.array_equal(sa["pos"], sb["pos"])
    for x, y in zip(ga, gb):
        assert np.array_equal(x, y)
    # a term is the same FP32 number in either order; blocks of 32 are summed
    # in FP32 (at most 32 roundings of 2^-24 of the block's terms), the blocks
    # with compensation: 34 covers both and the FP64 sums
    light = sa["mass"] < np.sort(sa["mass"])[-16]
    ends = [int(first[g]), int(first[g + 1]), 0, n // 2, n - 1]
    for i in sorted(set(list(range(ends[0], ends[1])) + ends[2:])):
        d = sa["pos"] - sa["pos"][i]
        r2 = (d * d).sum(1)
        ok = light & (r2 > 0)
        terms = (bh.G * sa["mass"][ok] / r2[ok]).sum()
        assert np.abs(sa["acc"][i] - sb["acc"][i]).max() <= 2 * 34 * 2.0**-24 * 2 * terms
