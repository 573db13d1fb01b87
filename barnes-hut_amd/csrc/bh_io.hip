// bh_io.hip -- bodies between the caller's arrays and the device.
//
// The caller's vectors are arrays of (x, y, z), the device keeps one array per
// component: both conversions run on the device, from and to a staging area,
// so that host memory is only ever copied in whole runs.  The heavy set (the
// kMaxHeavy most massive bodies of every system, ties by row, ranked by row)
// is chosen on the device too.  (On the host the conversions, the selection's
// index sort and three arrays of per-body defaults took 5 of the 7 ms of an
// upload of 300,149 bodies.)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bh_internal.hpp"

namespace bh {
namespace {

constexpr int kNT = 256;

// The triples v[3 i + a] into component arrays.
__global__ __launch_bounds__(kNT) void k_split3(const double* __restrict__ v, size_t n, double* __restrict__ x,
                                                double* __restrict__ y, double* __restrict__ z)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (i >= n) return;
    x[i] = v[3 * i];
    y[i] = v[3 * i + 1];
    z[i] = v[3 * i + 2];
}

// The parts of the bodies that the caller asked for (others null), each a run
// of the staging area.
__global__ __launch_bounds__(kNT) void k_pack(Bodies b, size_t n, PackedBodies out)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (i >= n) return;
    if (out.pos) {
        out.pos[3 * i] = b.px[i];
        out.pos[3 * i + 1] = b.py[i];
        out.pos[3 * i + 2] = b.pz[i];
    }
    if (out.vel) {
        out.vel[3 * i] = b.vx[i];
        out.vel[3 * i + 1] = b.vy[i];
        out.vel[3 * i + 2] = b.vz[i];
    }
    if (out.acc) {
        out.acc[3 * i] = b.ax[i];
        out.acc[3 * i + 1] = b.ay[i];
        out.acc[3 * i + 2] = b.az[i];
    }
    if (out.mass) out.mass[i] = b.m[i];
    if (out.ids) out.ids[i] = b.id[i];
}

// No previous walk, no accelerations; ids in row order unless they were given.
__global__ __launch_bounds__(kNT) void k_new_bodies(Bodies b, size_t n, int own_ids)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (i >= n) return;
    b.pcost[i] = 0u;
    b.ax[i] = 0.0;
    b.ay[i] = 0.0;
    b.az[i] = 0.0;
    if (own_ids) b.id[i] = i;
}

// ------------------------------------------------------------- heavy set
// Bodies in order of descending mass, then of ascending row.
struct Pick {
    double m;
    uint32_t i;   // row; kNoRow: none
};
constexpr uint32_t kNoRow = 0xffffffffu;

__device__ inline bool heavier(const Pick& a, const Pick& b)
{
    if (a.i == kNoRow || b.i == kNoRow) return b.i == kNoRow && a.i != kNoRow;
    return a.m > b.m || (!(b.m > a.m) && a.i < b.i);
}

// The heaviest of the block's picks, in every thread.
__device__ inline Pick block_heaviest(Pick p)
{
    __shared__ Pick s[kNT / 64];
    for (int o = 32; o > 0; o >>= 1) {
        const Pick q{__shfl_xor(p.m, o, 64), static_cast<uint32_t>(__shfl_xor(static_cast<int>(p.i), o, 64))};
        if (heavier(q, p)) p = q;
    }
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = p;
    __syncthreads();
    p = s[0];
    for (int k = 1; k < kNT / 64; ++k)
        if (heavier(s[k], p)) p = s[k];
    __syncthreads();
    return p;
}

// Candidates of one run of kHeavyRun rows: its kMaxHeavy heaviest, in order.
// A thread holds its rows' masses in registers; each round it offers its
// heaviest row that was not taken (rows are taken at most once).
constexpr uint32_t kPerThread = kHeavyRun / kNT;

__global__ __launch_bounds__(kNT) void k_heavy_candidates(const double* __restrict__ m, TreeBuffers tb,
                                                          const uint32_t* __restrict__ run_sys,
                                                          Pick* __restrict__ cand)
{
    const SysScalars* sy = tb.sys + run_sys[2 * blockIdx.x];
    const uint32_t lo = sy->body_lo + run_sys[2 * blockIdx.x + 1] * kHeavyRun;
    const uint32_t hi = min(sy->body_hi, lo + kHeavyRun);
    double v[kPerThread];
    uint32_t free_rows = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPerThread; ++k) {
        const uint32_t i = lo + k * kNT + threadIdx.x;
        v[k] = i < hi ? m[i] : 0.0;
        if (i < hi) free_rows |= 1u << k;
    }
    for (int r = 0; r < kMaxHeavy; ++r) {
        Pick p{0.0, kNoRow};
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const Pick q{v[k], (free_rows >> k) & 1u ? lo + k * kNT + threadIdx.x : kNoRow};
            if (heavier(q, p)) p = q;
        }
        const Pick best = block_heaviest(p);
        if (best.i != kNoRow && (best.i - lo) % kNT == threadIdx.x) free_rows &= ~(1u << ((best.i - lo) / kNT));
        if (threadIdx.x == 0) cand[static_cast<size_t>(blockIdx.x) * kMaxHeavy + r] = best;
    }
}

// One block per system: the heaviest of its runs' candidates (each run's are
// in order, so a run offers its first that was not taken), ranked by row.
__global__ __launch_bounds__(kNT) void k_heavy_pick(Bodies b, TreeBuffers tb, const uint32_t* __restrict__ sys_run,
                                                    const Pick* __restrict__ cand)
{
    __shared__ uint32_t rows[kMaxHeavy];
    const uint32_t s = blockIdx.x, r0 = sys_run[s], r1 = sys_run[s + 1];
    const uint32_t nh = tb.sys[s].n_heavy;
    Pick last{0.0, kNoRow};
    for (uint32_t r = 0; r < nh; ++r) {
        Pick p{0.0, kNoRow};
        for (uint32_t run = r0 + threadIdx.x; run < r1; run += kNT) {
            const Pick* c = cand + static_cast<size_t>(run) * kMaxHeavy;
            for (int k = 0; k < kMaxHeavy; ++k) {   // its first after the last one taken
                const Pick q = c[k];
                if (r > 0 && !heavier(last, q)) continue;
                if (heavier(q, p)) p = q;
                break;
            }
        }
        last = block_heaviest(p);
        if (threadIdx.x == 0) rows[r] = last.i;
    }
    __syncthreads();
    if (threadIdx.x < nh && rows[threadIdx.x] != kNoRow) {
        uint32_t rank = 0;
        for (uint32_t k = 0; k < nh; ++k) rank += rows[k] < rows[threadIdx.x] ? 1u : 0u;
        b.hrank[rows[threadIdx.x]] = static_cast<int8_t>(rank);
    }
}

// The system of every row (runs of rows of one system) and no heavy rank yet.
__global__ __launch_bounds__(kNT) void k_row_systems(Bodies b, TreeBuffers tb, const uint32_t* __restrict__ run_sys,
                                                     uint8_t* __restrict__ bsys)
{
    const uint32_t s = run_sys[2 * blockIdx.x];
    const uint32_t lo = tb.sys[s].body_lo + run_sys[2 * blockIdx.x + 1] * kHeavyRun;
    const uint32_t hi = min(tb.sys[s].body_hi, lo + kHeavyRun);
    for (uint32_t i = lo + threadIdx.x; i < hi; i += kNT) {
        bsys[i] = static_cast<uint8_t>(s);
        b.hrank[i] = -1;
    }
}

inline unsigned nblk(size_t n) { return static_cast<unsigned>((n + kNT - 1) / kNT); }

}  // namespace

size_t heavy_scratch_bytes(uint32_t n_runs) { return sizeof(Pick) * kMaxHeavy * static_cast<size_t>(n_runs); }

void launch_split3(const double* v, size_t n, double* x, double* y, double* z, hipStream_t s)
{
    if (n) k_split3<<<nblk(n), kNT, 0, s>>>(v, n, x, y, z);
}

void launch_pack(const Bodies& b, size_t n, const PackedBodies& out, hipStream_t s)
{
    if (n) k_pack<<<nblk(n), kNT, 0, s>>>(b, n, out);
}

void launch_new_bodies(const Bodies& b, size_t n, bool own_ids, hipStream_t s)
{
    if (n) k_new_bodies<<<nblk(n), kNT, 0, s>>>(b, n, own_ids ? 1 : 0);
}

void launch_heavy_set(const Bodies& b, const TreeBuffers& tb, const uint32_t* run_sys, uint32_t n_runs,
                      const uint32_t* sys_run, uint8_t* bsys, void* scratch, hipStream_t s)
{
    if (n_runs == 0) return;
    Pick* cand = static_cast<Pick*>(scratch);
    k_row_systems<<<n_runs, kNT, 0, s>>>(b, tb, run_sys, bsys);
    k_heavy_candidates<<<n_runs, kNT, 0, s>>>(b.m, tb, run_sys, cand);
    k_heavy_pick<<<tb.n_sys, kNT, 0, s>>>(b, tb, sys_run, cand);
}

}  // namespace bh
