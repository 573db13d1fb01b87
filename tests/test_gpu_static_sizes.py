"""GPU test of the plain form's small sizes: the static evaluation sorts with
the merge sort alone, whose rounds end in one or the other buffer (one tile to
2,048 keys, one round to 32,768, two above), and sums a small tree's moments in
one workgroup.  Bits equal a context's evaluation with the radix sort and one
moment launch per depth, whatever the input order and with equal keys."""
import sys

import numpy as np
import pytest

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n", [1, 2, 65, 2047, 2048, 2049, 4096, 4097, 32767, 32768, 32769, 65535, 65536])
def test_static_sizes_match_full_sort_and_levels(bh, n):
    say("static evaluation", n, "bodies")
    rng = np.random.default_rng(n)
    pos, vel, m = (a[:n] for a in bh.generate(bh.GEN_TROJAN, 7, max(n, 65)))
    order = rng.permutation(n)
    pos, m = pos[order].copy(), m[order].copy()
    if n > 2000:   # equal keys, within a tile and across tiles
        pos[rng.integers(0, n, 300)] = pos[5]
        pos[n - 9:] = pos[17]
    with bh.Engine(theta=0.9) as e:
        e.set_sort_mode(bh.SORT_FULL)
        e.set_moment_cutoff(21)
        e.set_bodies(pos, np.zeros_like(pos), m)
        e.compute_accelerations(theta=0.9)
        st = e.get_bodies()
    want = np.empty_like(pos)
    want[st["ids"].astype(np.int64)] = st["acc"]
    hip = Hip(bh)
    try:
        dpos, dm, dacc = hip.put(pos), hip.put(m), hip.put(np.full((n, 3), np.nan))
        rc = bh.load().bh_compute_accelerations_static(n, dpos, dm, 0.9, bh.G, 0.0, dacc, None)
        assert rc == 0, bh.load().bh_static_last_error()
        hip.sync()
        got = hip.get(dacc, (n, 3))
    finally:
        hip.free()
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
