"""GPU test of the plain walk by one wavefront per body (small systems) at the
sizes and lists where it can go wrong: part-filled wavefronts and blocks, lists
of a few, of one chunk of 64, and longer than the ordered list's buffer (small
theta), equal keys, massless bodies, and both sides of the sizes at which the
per-lane walk takes over.  Bits equal the oracle's."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n,theta", [
    (2, 1.05), (3, 0.0), (5, 1.05), (63, 0.0), (64, 0.0), (65, 0.0), (66, 0.0), (129, 0.0), (1535, 0.0), (1537, 0.0),
    (1538, 0.0), (3001, 0.05), (3001, 1.05), (4098, 0.4), (16384, 2.0), (16385, 2.0), (20480, 0.3), (20480, 1.2),
    (20480, 1.21), (20481, 1.05)])
@pytest.mark.parametrize("odd", [False, True])
def test_small_walk_matches_oracle(bh, orc, n, theta, odd):
    say("plain walk", n, "bodies, theta", theta, "equal keys and massless" if odd else "")
    pos, vel, m = (a[:n].copy() for a in bh.generate(bh.GEN_TROJAN, 11, max(n, 65)))
    if odd:
        k = max(1, n // 10)
        pos[:k] = pos[n - 1]
        m[k // 2:2 * k] = 0.0
    soft2 = 1e-9 if odd else 0.0
    with bh.Engine(theta=theta) as e:
        e.set_bodies(pos, vel, m)
        acc = e.compute_accelerations(theta=theta, soft2=soft2)
        ids = e.get_bodies()["ids"]
    want = orc.force_path(pos, m, theta=theta, soft2=soft2)
    assert np.array_equal(ids, want["ids"])
    assert np.array_equal(acc.view(np.uint64), want["acc"].view(np.uint64))
