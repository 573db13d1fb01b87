"""GPU test of the bodies' way to the device and back: uploads and downloads at
the edges of the chunks (4 MiB of packed bodies) and of the threaded copies,
every subset of the outputs, and the heavy set chosen on the device (ties by
row, ranks by row, several runs of rows and several systems)."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


# 88 bytes a body: one chunk holds 47,662 bodies
@pytest.mark.parametrize("n", [1, 2, 4095, 4097, 47662, 47663, 130001])
def test_bodies_come_back_as_they_went(bh, n):
    say("transfer", n)
    rng = np.random.default_rng(n)
    pos, vel, mass = rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.random(n)
    ids = rng.permutation(n).astype(np.uint64) + 5
    with bh.Engine() as e:
        for given in (ids, None):
            e.set_bodies(pos, vel, mass, given)
            s = e.get_bodies()
            want = np.arange(n, dtype=np.uint64) if given is None else given
            for a, b in ((s["pos"], pos), (s["vel"], vel), (s["mass"], mass), (s["acc"], 0 * pos)):
                assert np.array_equal(a, b)
            assert np.array_equal(s["ids"], want)
        # any output may be left out
        for mask in range(32):
            out = [np.full(sh, -1.0) for sh in ((n, 3), (n, 3), (n,), (n, 3))] + [np.zeros(n, np.uint64)]
            ptr = [a.ctypes.data_as(C.c_void_p) if mask >> k & 1 else None for k, a in enumerate(out)]
            assert e.lib.bh_get_bodies(e.h, ptr[0], ptr[1], ptr[2], ptr[4], ptr[3]) == 0
            for k, (a, b) in enumerate(zip(out, (pos, vel, mass, 0 * pos, np.arange(n, dtype=np.uint64)))):
                assert np.array_equal(a, b if mask >> k & 1 else (a * 0 - 1 if k < 4 else a * 0))


def heavy_reference(mass, off):
    """Rows of each system's 16 most massive bodies, ties by row."""
    out = []
    for lo, hi in zip(off[:-1], off[1:]):
        order = sorted(range(lo, hi), key=lambda i: (-mass[i], i))
        out.append(sorted(order[:16]))
    return out


@pytest.mark.parametrize("sizes", [[1], [16], [17, 3], [5000, 9, 12289, 700]])
@pytest.mark.parametrize("levels", [1, 3, 1000000])
def test_heavy_set(bh, sizes, levels):
    """The heavy bodies have their accelerations summed directly in FP64 and
    agree with the direct sum; light ones carry the tree's and FP32's errors."""
    say("heavy", sizes, levels)
    n = sum(sizes)
    off = np.concatenate([[0], np.cumsum(sizes)])
    rng = np.random.default_rng(n)
    pos, vel = rng.normal(size=(n, 3)), np.zeros((n, 3))
    mass = 1e24 * (1.0 + rng.integers(0, levels, n) / levels)
    with bh.Engine(form=bh.FORM_MIXED, theta=0.7) as e:
        e.set_bodies(pos, vel, mass)
        if len(sizes) > 1:
            e.set_systems(sizes)
        acc = e.compute_accelerations(bh.FORM_MIXED, 0.7)
        s = e.get_bodies()
        ids = s["ids"].astype(np.int64)
        ds = e.direct_sum(np.arange(n))
    err = np.linalg.norm(acc - ds, axis=1) / np.linalg.norm(ds, axis=1).clip(1e-300)
    exact = np.zeros(n, bool)
    exact[ids] = err <= 1e-13
    for rows, lo, hi in zip(heavy_reference(mass, off), off[:-1], off[1:]):
        assert exact[rows].all()
        if hi - lo > 2000:     # light bodies carry FP32 sums
            light = np.setdiff1d(np.arange(lo, hi), rows)
            assert exact[light].mean() < 0.1
