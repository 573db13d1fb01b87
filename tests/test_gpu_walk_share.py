"""GPU test of the mixed walk's two ways of walking a group: by one wavefront
and by the four of a block.  With walk_blocks = 1 a system of more than two
groups is walked by lone wavefronts; with the default grid a small system's
groups are shared in the first evaluation, and later those listed as costly
are (key order: a list; cost order: the first of the order).  Every way gives
the same bits, lists and work."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 24.0


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


def bodies(bh, n, coincident):
    pos, vel, mass = bh.generate(bh.GEN_TROJAN if n > 2000 else bh.GEN_BELT, 5, n)
    if coincident:
        # co-keyed leaves of 300, 20 and 9 bodies, and one with heavy bodies
        for lo, hi in ((100, 400), (1000, 1020), (1500, 1509)):
            pos[lo:hi] = pos[lo]
            vel[lo:hi] = vel[lo]
        pos[40:45] = pos[2]
    return pos, vel, mass


def walk(bh, data, theta, gmax, sched, blocks):
    """Accelerations, ids and per-group figures of a first evaluation and of
    two steps after it (the second with a previous walk's work)."""
    out = []
    with bh.Engine(form=bh.FORM_MIXED, theta=theta) as e:
        e.set_bodies(*data)
        e.set_schedule(sched)
        e.set_group_params(gmax, 2.0, 32, blocks)
        for _ in range(3):
            e.step(1, DT)
            s = e.get_bodies()
            first, inter, visit = e.groups()
            out.append((s["acc"].view(np.uint64), s["ids"], first, inter, visit, e.group_work()))
    return out


@pytest.mark.parametrize("n,coincident,gmax,theta", [
    (9, False, 64, 1.05),        # one group, fewer light bodies than a wavefront
    (65, False, 64, 1.05),
    (700, False, 1, 1.05),       # groups of one body: 32 shares
    (700, False, 64, 0.5),       # no relative opening test
    (5000, True, 64, 1.05),      # leaves of more than 8 bodies take turns
    (5000, True, 17, 0.6),
    (30011, False, 64, 1.05),    # more groups than blocks
])
def test_shared_and_lone_walks_agree(bh, n, coincident, gmax, theta):
    data = bodies(bh, n, coincident)
    for sched in (bh.SCHED_KEY_ORDER, bh.SCHED_PREV_COST):
        say("walk_share", n, coincident, gmax, theta, sched)
        lone = walk(bh, data, theta, gmax, sched, 1)
        shared = walk(bh, data, theta, gmax, sched, 0)
        for step, (a, b) in enumerate(zip(lone, shared)):
            for x, y in zip(a, b):
                assert np.array_equal(x, y), f"step {step}"
