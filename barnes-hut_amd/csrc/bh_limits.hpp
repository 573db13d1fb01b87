// bh_limits.hpp -- sizes that host code checks against buffers, free of HIP.
#pragma once

#include <cstddef>
#include <cstdint>

#include "bh_pick.hpp"

namespace bh {

constexpr int kMaxHeavy = 16;     // bodies per system summed directly in FP64 by the mixed forms
constexpr int kMaxSystems = 256;  // systems per context (the sort's system pass uses 8-bit digits)

// The heavy set is chosen over runs of at most kHeavyRun rows of one system,
// each of which leaves kMaxHeavy candidates (Pick) in a scratch area.
constexpr uint32_t kHeavyRun = 4096;

// a system of k bodies has ceil(k / kHeavyRun) <= k / kHeavyRun + 1 runs
constexpr size_t max_heavy_runs(size_t n) { return n / kHeavyRun + kMaxSystems; }
constexpr size_t heavy_scratch_bytes(size_t n_runs) { return sizeof(Pick) * kMaxHeavy * n_runs; }

// Staging area of the host transfers and the heavy set's scratch, for up to n
// bodies: 96 bytes a body (the light boxes of 2 n nodes, in whose place it
// lies; a packed body takes 88), and at least the candidates of every run.
// One-body systems have 256 bytes of candidates a body.
constexpr size_t staging_doubles(size_t n)
{
    const size_t boxes = 12 * n, runs = heavy_scratch_bytes(max_heavy_runs(n)) / sizeof(double);
    return boxes > runs ? boxes : runs;
}

}  // namespace bh
