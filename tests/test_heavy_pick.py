"""The order in which the heavy set is chosen, and its selection where that order
decides most: masses that are no numbers, infinite, zero or equal, and rows laid
out so that the first cut leaves too many to be ranked by counting."""
import pathlib
import shutil
import subprocess
import sys

import numpy as np
import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

DRIVER = r"""
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>
#include "bh_pick.hpp"
// as the device ranks a set: how many are heavier
static bool ranks_are_a_permutation(const std::vector<bh::Pick>& v)
{
    std::vector<int> taken(v.size(), 0);
    for (const bh::Pick& a : v) {
        size_t rank = 0;
        for (const bh::Pick& b : v) rank += bh::heavier(b, a);
        if (rank >= v.size() || taken[rank]++) return false;
    }
    return true;
}
int main()
{
    const double some[] = {NAN, -NAN, INFINITY, -INFINITY, 0.0, -0.0, 1.0, 2.0, -1.0, 1e300, 5e-324};
    std::mt19937 rng(3);
    for (int trial = 0; trial < 400; ++trial) {
        std::vector<bh::Pick> v;
        for (uint32_t i = 0; i < 40; ++i)
            v.push_back(bh::pick(trial % 2 ? some[rng() % 11] : (rng() % 9 ? static_cast<double>(rng()) : NAN), i));
        if (!ranks_are_a_permutation(v)) return std::printf("trial %d\n", trial), 1;
    }
    if (bh::heavier(bh::pick(1.0, 3), bh::pick(1.0, 2)) || !bh::heavier(bh::pick(-INFINITY, 0), bh::Pick{9.0, bh::kNoRow}) ||
        !bh::heavier(bh::pick(-1e300, 1), bh::pick(NAN, 0)) || bh::heavier(bh::pick(-0.0, 1), bh::pick(0.0, 0)))
        return std::puts("order"), 1;
    std::puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_ranks_by_counting_are_all_different(tmp_path):
    src, exe = tmp_path / "pick.cpp", tmp_path / "pick"
    src.write_text(DRIVER)
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(ROOT / "barnes-hut_amd" / "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


def bodies(n, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(n, 3)), np.zeros((n, 3)), 1e24 * (1.0 + rng.random(n))


def forces(bh, pos, vel, mass, sizes=None):
    with bh.Engine(form=bh.FORM_MIXED, theta=0.7) as e:
        e.set_bodies(pos, vel, mass)
        if sizes:
            e.set_systems(sizes)
        acc = e.compute_accelerations(bh.FORM_MIXED, 0.7)
        s = e.get_bodies()
        return acc, s, e.direct_sum(np.arange(len(mass)))


@pytest.mark.gpu
@pytest.mark.parametrize("share", [0.001, 0.3, 1.0])
def test_system_beside_one_with_nan_masses(bh, share):
    """A system whose masses are partly no numbers leaves its neighbours alone."""
    say("nan masses", share)
    sizes = [3000, 9000, 12, 700]
    pos, vel, mass = bodies(sum(sizes), 5)
    clean = mass.copy()
    bad = np.random.default_rng(6).random(9000) < share
    mass[3000:12000][bad] = np.nan
    acc, s, _ = forces(bh, pos, vel, mass, sizes)
    want, w, _ = forces(bh, pos, vel, clean, sizes)
    keep = np.r_[0:3000, 12000:sum(sizes)]
    assert np.array_equal(s["ids"], w["ids"])
    assert np.array_equal(acc[keep].view(np.uint64), want[keep].view(np.uint64))
    assert np.array_equal(np.isnan(s["mass"]), np.isnan(mass)[s["ids"].astype(np.int64)])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1024 + 256, 4096, 5000, 3 * 4096 + 17])
def test_rows_of_one_set_light(bh, n):
    """Of every 256 rows 16 are light: the first cut keeps all the others, more
    than are ranked by counting."""
    say("rows of one set light", n)
    pos, vel, mass = bodies(n, n)
    mass[np.arange(n) % 256 < 16] *= 1e-6
    acc, s, direct = forces(bh, pos, vel, mass)
    ids = s["ids"].astype(np.int64)
    err = np.empty(n)
    err[ids] = np.linalg.norm(acc - direct, axis=1) / np.linalg.norm(direct, axis=1)
    heavy = sorted(range(n), key=lambda i: (-mass[i], i))[:16]
    assert err[heavy].max() <= 1e-13
    assert (np.delete(err, heavy) <= 1e-13).mean() < 0.1     # light bodies carry FP32 sums
