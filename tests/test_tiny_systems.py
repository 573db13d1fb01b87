"""Ensembles of systems of a body or two.  Every system has at least one run of
rows in the selection of the heavy set, and a run's candidates take 256 bytes:
more than a body's share of the staging area, which has to be sized for both."""
import pathlib
import shutil
import subprocess
import sys

import numpy as np
import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

DRIVER = r"""
#include <algorithm>
#include <cstdio>
#include "bh_limits.hpp"
// systems of `size` bodies (the last takes the rest): their runs and candidates fit
static bool fits(size_t n, size_t systems)
{
    const size_t size = n / systems;
    size_t runs = 0;
    for (size_t s = 0; s < systems; ++s)
        runs += (std::max<size_t>(s + 1 < systems ? size : n - size * (systems - 1), 1) + bh::kHeavyRun - 1) / bh::kHeavyRun;
    const size_t cap = std::max<size_t>(n, 64);   // the buffers' smallest capacity
    return runs <= bh::max_heavy_runs(cap) && bh::heavy_scratch_bytes(runs) <= 8 * bh::staging_doubles(cap) &&
           88 * n <= 8 * bh::staging_doubles(cap);
}
int main()
{
    const size_t sizes[] = {1, 2, 3, 700, bh::kHeavyRun - 1, bh::kHeavyRun, bh::kHeavyRun + 1, 100003};
    for (size_t systems = 1; systems <= static_cast<size_t>(bh::kMaxSystems); ++systems)
        for (size_t k : sizes)
            for (size_t rest : {size_t{0}, size_t{1}, systems - 1})
                if (!fits(k * systems + rest, systems)) return std::printf("%zu systems of %zu + %zu\n", systems, k, rest), 1;
    std::puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_candidates_fit_the_staging_area(tmp_path):
    src, exe = tmp_path / "limits.cpp", tmp_path / "limits"
    src.write_text(DRIVER)
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(ROOT / "barnes-hut_amd" / "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1] * 64, [2] * 64, [2] * 100, [1] * 256, [2] * 256, [1, 17] * 20])
def test_forces_of_tiny_systems(bh, sizes):
    """Up to 16 bodies are all heavy: their accelerations are the direct sums."""
    print("[gpu-case] tiny systems", len(sizes), sizes[:2], file=sys.stderr, flush=True)
    n = sum(sizes)
    rng = np.random.default_rng(n)
    pos, vel, mass = rng.normal(size=(n, 3)), np.zeros((n, 3)), 1e24 * (1.0 + rng.random(n))
    with bh.Engine(form=bh.FORM_MIXED, theta=0.7) as e:
        e.set_bodies(pos, vel, mass)
        e.set_systems(sizes)
        acc = e.compute_accelerations(bh.FORM_MIXED, 0.7)
        s = e.get_bodies()
        direct = e.direct_sum(np.arange(n))
    off = np.concatenate([[0], np.cumsum(sizes)])
    for lo, hi in zip(off[:-1], off[1:]):   # a system keeps its rows
        assert np.array_equal(np.sort(s["ids"][lo:hi]), np.arange(lo, hi, dtype=np.uint64))
        if hi - lo <= 16:
            scale = np.linalg.norm(direct[lo:hi], axis=1).max()
            assert np.abs(acc[lo:hi] - direct[lo:hi]).max() <= 1e-13 * scale
    assert np.array_equal(s["mass"], mass[s["ids"].astype(np.int64)])
