"""GPU test of the mixed walk's timeline: a worker wave walks one group at a
time, so the spans of the groups with the same worker index do not overlap, and
the groups of a walk with many of them are spread over a block's four waves."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 24.0


@pytest.mark.parametrize("n,blocks", [(3000, 0), (60000, 0), (60000, 7), (200000, 0)])
def test_a_worker_walks_one_group_at_a_time(bh, n, blocks):
    data = bh.generate(bh.GEN_TROJAN, 3, n)
    for sched in (bh.SCHED_KEY_ORDER, bh.SCHED_PREV_COST):
        print("[gpu-case] timeline", n, blocks, sched, file=sys.stderr, flush=True)
        with bh.Engine(form=bh.FORM_MIXED, theta=1.05) as e:
            e.set_bodies(*data)
            e.set_schedule(sched)
            e.set_group_params(64, 2.0, 32, blocks)
            e.step(2, DT)
            start, end, worker = e.group_timeline()
            waves = 4 * e.group_params()["walk_blocks"]
        assert (end >= start).all() and worker.max() < waves
        order = np.lexsort((start, worker))
        same = worker[order][1:] == worker[order][:-1]
        assert (start[order][1:] >= end[order][:-1])[same].all()
        if len(worker) > 8 * waves:   # lone waves take most groups: every wave has some
            assert len(np.unique(worker)) == waves
