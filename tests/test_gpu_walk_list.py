"""GPU test of the list of shared groups at its end.  After a walk with groups of
up to 64 bodies a step with groups of one body has many more groups, each with
the work that its body's old group took, so more of them exceed the sharing limit
than the list holds: the listed ones are shared, the others walked alone, each
once.  The split schedule shares none and gives the same bits."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 24.0
LIST = 65536   # entries of the list


def over_the_limit(e):
    """Bodies whose group's work exceeds the sharing limit of the next walk."""
    first, _, _ = e.groups()
    work = e.group_work().astype(object)
    waves = 4 * e.group_params()["walk_blocks"]
    total, groups = int(sum(work)), len(work)
    many = total * groups * 3 // (waves * waves * 5)
    limit = min(many, max(total // waves // 8, 4 * (total // groups)))
    return int(np.diff(first)[np.array([w > limit for w in work])].sum())


@pytest.mark.parametrize("n", [150001])
def test_more_groups_over_the_limit_than_the_list_holds(bh, n):
    print("[gpu-case] walk list", n, file=sys.stderr, flush=True)
    data = bh.generate(bh.GEN_BELT, 5, n)
    out = []
    for shared in (False, True):
        with bh.Engine(form=bh.FORM_MIXED, theta=1.05) as e:
            e.set_graph(False)
            e.set_bodies(*data)
            if not shared:
                e.set_schedule(bh.SCHED_PREV_COST)
                e.set_schedule_split(4)
            e.step(1, DT)
            assert over_the_limit(e) > LIST
            e.set_group_params(1, 2.0, 32, 0)
            e.step(1, DT)
            assert len(e.groups()[1]) == n
            s = e.get_bodies()
            e.step(1, DT)
            out.append((s, e.get_bodies()))
    for a, b in zip(*out):
        for k in ("pos", "vel", "acc", "ids"):
            assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64)), k
