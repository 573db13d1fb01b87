"""GPU test of the direct sum's blocks of 1, 2 and 4 samples: every sample's
accelerations have the same bits however many samples share its block, across
systems and with co-located bodies, and agree with a
plain FP64 sum."""
import math
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("m", [1, 3, 1023, 1024, 1027, 4096, 4099])
@pytest.mark.parametrize("systems", [None, [700, 9, 1500, 791]])
def test_samples_do_not_depend_on_their_block(bh, m, systems):
    say("direct", m, systems)
    n = 3000
    pos, vel, mass = bh.generate(bh.GEN_BELT, 11, n)
    pos[50:60] = pos[50]          # co-located bodies add nothing to each other
    rng = np.random.default_rng(m)
    idx = rng.integers(0, n, m)   # repeated samples are allowed
    soft2 = 1e-8 if m % 2 else 0.0
    with bh.Engine() as e:
        e.set_bodies(pos, vel, mass)
        if systems:
            e.set_systems(systems)
        acc = e.direct_sum(idx, soft2=soft2)
        # blocks of one sample
        alone = np.concatenate([e.direct_sum(idx[k:k + 500], soft2=soft2) for k in range(0, m, 500)])
    assert np.array_equal(acc.view(np.uint64), alone.view(np.uint64))
    # each term has a relative error of a few 2^-53, the compensated sums less:
    # 1e-14 of the sum of the terms' sizes
    off = np.concatenate([[0], np.cumsum(systems or [n])])
    for k in range(0, m, max(1, m // 20)):
        s = int(np.searchsorted(off, idx[k], side="right")) - 1
        lo, hi = off[s], off[s + 1]
        d = pos[lo:hi] - pos[idx[k]]
        r2 = (d * d).sum(1) + soft2
        f = np.where(((d * d).sum(1) > 0) & (np.arange(lo, hi) != idx[k]), bh.G * mass[lo:hi] / np.where(r2 > 0, r2, 1) ** 1.5, 0)
        t = f[:, None] * d
        exact = np.array([math.fsum(t[:, a]) for a in range(3)])   # numpy's own sum is off by more
        assert np.all(np.abs(exact - acc[k]) <= 1e-14 * np.abs(t).sum(0))
