"""GPU test of the plain walk whose lanes wait for their wavefront's last one, at
the sizes where the limit changes and with a part-filled last wavefront: bits
equal those of the counting walk, which has no limit."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n,theta", [(99999, 1.05), (100001, 1.05), (159999, 0.6), (160000, 0.79), (160063, 1.05),
                                     (200001, 0.4), (262145, 3.0)])
def test_limited_lead_matches_counting_walk(bh, n, theta):
    say("walk lead", n, theta)
    pos, vel, m = bh.generate(bh.GEN_TROJAN, 13, n)
    pos[1000:1100] = pos[500]   # equal keys
    m[2000:2050] = 0.0
    out = []
    for counting in (False, True):
        with bh.Engine(theta=theta) as e:
            e.set_counting(counting)
            e.set_bodies(pos, vel, m)
            out.append(e.compute_accelerations(theta=theta, soft2=1e-12))
    assert np.array_equal(out[0].view(np.uint64), out[1].view(np.uint64))
