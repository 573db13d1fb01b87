"""GPU test of a context whose last upload found no room on the device: the
bodies before are gone, so every call that would launch on them says so, and the
next upload that fits works as if nothing had been."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOO_MANY = 1 << 30   # about 1.2 TB of buffers


def test_calls_after_an_upload_without_room(bh):
    print("[gpu-case] no room", file=sys.stderr, flush=True)
    data = bh.generate(bh.GEN_BELT, 5, 3000)
    with bh.Engine(form=bh.FORM_MIXED, theta=1.05) as e:
        def run():
            e.set_bodies(*data)
            e.step(2, 1.0 / 24.0)
            return e.get_bodies()

        want = run()
        # (fails before it reads the arrays; one upload only: taking all of the
        # device's memory lasts seconds)
        p = [a.ctypes.data_as(C.c_void_p) for a in data]
        assert e.lib.bh_set_bodies(e.h, TOO_MANY, *p, None) == bh.ERR_NOMEM
        out = np.full((3000, 3), 7.0)
        o = out.ctypes.data_as(C.c_void_p)
        assert e.lib.bh_get_bodies(e.h, o, None, None, None, None) == bh.ERR_STATE
        for form in (bh.FORM_PLAIN, bh.FORM_MIXED):
            assert e.lib.bh_compute_accelerations(e.h, form, 1.05, bh.G, 0.0, o) == bh.ERR_STATE
        assert e.lib.bh_step(e.h, 1, 1.0 / 24.0) == bh.ERR_STATE
        sizes = np.array([1000, 2000], np.int64)
        assert e.lib.bh_set_systems(e.h, 2, sizes.ctypes.data_as(C.c_void_p)) == bh.ERR_STATE
        idx = np.zeros(1, np.int64)
        assert e.lib.bh_direct_sum(e.h, 1, idx.ctypes.data_as(C.c_void_p), bh.G, 0.0, o) == bh.ERR_STATE
        assert (out == 7.0).all()
        again = run()
    for k in ("pos", "vel", "acc", "ids"):
        assert np.array_equal(again[k].view(np.uint64), want[k].view(np.uint64))


def test_transfers_after_an_error_of_the_caller(bh):
    """An error that the caller's own HIP calls left on the runtime's record does
    not make an upload or a download fail."""
    print("[gpu-case] error of the caller", file=sys.stderr, flush=True)
    hip = C.CDLL("libamdhip64.so.7")
    pos, vel, mass = bh.generate(bh.GEN_BELT, 5, 3000)
    with bh.Engine(form=bh.FORM_MIXED) as e:
        for call in (lambda: e.set_bodies(pos, vel, mass), lambda: e.set_systems([1000, 2000]), lambda: e.get_bodies()):
            assert hip.hipSetDevice(9999) != 0
            assert hip.hipPeekAtLastError() != 0
            s = call()
        assert np.array_equal(s["pos"], pos)
