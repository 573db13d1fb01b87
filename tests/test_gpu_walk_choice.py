"""GPU test of the plain walk's choice between one lane and one wavefront per body,
which looks at the length of a small system's lists: long ones (belts, small
theta), short ones (a Kuiper belt, a cube, clusters far apart, large theta) and
both sides of the sizes at which it begins and ends.  Bits equal the counting
walk's (one lane per body), replayed steps included, and short lists do not take
longer than those of a system just too large for the choice."""
import sys

import numpy as np
import pytest

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu
HOUR = 1.0 / 24.0


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def shape(bh, name, n):
    rng = np.random.default_rng(n)
    if name in ("belt", "kuiper"):
        return bh.generate(bh.GEN_BELT if name == "belt" else bh.GEN_KUIPER, 3, n)
    if name == "cube":
        pos = rng.random((n, 3))
    else:
        pos = 100.0 * rng.normal(size=(8, 3))[rng.integers(0, 8, n)] + rng.normal(size=(n, 3))
        pos[: n // 10] = pos[n - 1]   # equal keys
    mass = 1e20 * rng.random(n)
    mass[: n // 20] = 0.0
    return pos, np.zeros((n, 3)), mass


@pytest.mark.parametrize("name", ["belt", "kuiper", "cube", "clusters"])
@pytest.mark.parametrize("n", [5500, 5501, 8192, 16385, 20479, 20480, 20481])
def test_bits_of_either_walk(bh, name, n):
    data = shape(bh, name, n)
    for theta in (0.4, 1.05, 3.0):
        say("walk choice", name, n, theta)
        out = []
        for counting in (False, True):
            with bh.Engine(theta=theta, soft2=1e-9) as e:
                e.set_counting(counting)
                e.set_bodies(*data)
                e.step(4, HOUR)   # replayed from the second on where nothing is counted
                out.append(e.get_bodies())
        for k in ("pos", "vel", "acc", "ids"):
            assert np.array_equal(bits(out[0][k]), bits(out[1][k])), (theta, k)


@pytest.mark.parametrize("name,theta", [("cube", 1.05), ("cube", 2.0), ("kuiper", 1.5), ("clusters", 3.0)])
def test_short_lists_are_walked_per_lane(bh, name, theta):
    took = []
    for n in (20480, 20481):   # by wavefronts the first takes 1.7 to 5 times as long
        say("short lists", name, n, theta)
        with bh.Engine(theta=theta) as e:
            e.set_bodies(*shape(bh, name, n))
            t = []
            for _ in range(15):
                e.compute_accelerations(theta=theta)
                t.append(e.phase_ms()[3])
            took.append(np.median(t))
    say("ms of the walk", took)
    assert took[0] <= 1.4 * took[1]


@pytest.mark.parametrize("name,n", [("cube", 12288), ("belt", 12288), ("clusters", 20480)])
def test_static_evaluation_chooses_too(bh, name, n):
    say("static walk choice", name, n)
    pos, vel, mass = shape(bh, name, n)
    with bh.Engine(theta=1.05) as e:
        e.set_counting(True)
        e.set_bodies(pos, vel, mass)
        e.compute_accelerations(theta=1.05)
        st = e.get_bodies()
    want = np.empty_like(pos)
    want[st["ids"].astype(np.int64)] = st["acc"]
    hip = Hip(bh)
    try:
        dpos, dm, dacc = hip.put(pos), hip.put(mass), hip.alloc(24 * n)
        for _ in range(2):
            assert bh.load().bh_compute_accelerations_static(n, dpos, dm, 1.05, bh.G, 0.0, dacc, None) == 0
            hip.sync()
            assert np.array_equal(bits(hip.get(dacc, (n, 3))), bits(want))
    finally:
        hip.free()
