"""GPU test of a large download where no pinned memory is to be had: the bodies
come through pageable memory.  A child process finds a hipHostMalloc in front of
the runtime's that refuses large requests."""
import pathlib
import shutil
import subprocess
import sys

import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")]
ROOT = pathlib.Path(__file__).resolve().parents[1]

SHIM = r"""
#include <dlfcn.h>
#include <cstddef>
static int refused;
extern "C" int hipHostMalloc(void** p, size_t bytes, unsigned flags)
{
    if (bytes >= (size_t{1} << 20)) return ++refused, 2;   // hipErrorOutOfMemory
    static auto real = reinterpret_cast<int (*)(void**, size_t, unsigned)>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipHostMalloc"));
    return real(p, bytes, flags);
}
extern "C" int shim_refused() { return refused; }
"""

CHILD = r"""
import ctypes, sys
import numpy as np
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import conftest
bh = conftest.load_bh()
n = 130001
rng = np.random.default_rng(n)
pos, vel, mass = rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.random(n)
with bh.Engine() as e:
    for _ in range(2):
        e.set_bodies(pos, vel, mass)
        s = e.get_bodies()
        for a, b in ((s["pos"], pos), (s["vel"], vel), (s["mass"], mass), (s["acc"], 0 * pos), (s["ids"], np.arange(n, dtype=np.uint64))):
            assert np.array_equal(a, b)
    e.set_bodies(pos, vel, mass)   # no error is left behind
    e.compute_accelerations(bh.FORM_PLAIN, 1.5)
print("ok", shim.shim_refused())
"""


def test_download_without_pinned_memory(tmp_path):
    print("[gpu-case] no pinned memory", file=sys.stderr, flush=True)
    src, lib = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    r = subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", str(src), "-o", str(lib), "-ldl"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib), str(ROOT / "tests")], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    word, refused = r.stdout.split()
    assert word == "ok" and int(refused) == 2   # each get_bodies once; the accelerations alone (3.1 MB) need no chunks
