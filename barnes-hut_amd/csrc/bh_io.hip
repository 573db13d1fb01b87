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

// The `want` (<= kMaxHeavy) heaviest of the block's rows, in order, into
// out[0, want) (kNoRow past the last): each thread has a share of the rows,
// which rows(f) shows to f.  The heaviest rows of the block's kMaxHeavy sets of
// 16 threads are kMaxHeavy rows, so a row less heavy than all of them is not
// wanted; the others, some fifty of rows in no order, are gathered in LDS and
// ranked by counting.  (Taking the heaviest row 16 times, with a reduction over
// the block each, the two kernels below took 46 and 40 us at 19,054 bodies, now
// 21 each.)  Only if more than kGather are left are they taken one by one.
constexpr uint32_t kGather = 1024;
static_assert(kNT == 16 * kMaxHeavy, "kMaxHeavy sets of 16 threads");

template <typename Rows>
__device__ inline void block_top(uint32_t want, Rows rows, Pick* out)
{
    __shared__ Pick top[kMaxHeavy], some[kGather];
    __shared__ uint32_t n_some;
    Pick p{0.0, kNoRow};
    rows([&](const Pick& q) {
        if (heavier(q, p)) p = q;
    });
    for (int o = 8; o > 0; o >>= 1) {
        const Pick q{__shfl_xor(p.m, o, 64), static_cast<uint32_t>(__shfl_xor(static_cast<int>(p.i), o, 64))};
        if (heavier(q, p)) p = q;
    }
    if (threadIdx.x % 16 == 0) top[threadIdx.x / 16] = p;
    if (threadIdx.x == 0) n_some = 0;
    __syncthreads();
    Pick limit = top[0];   // (no row: a set without rows, then every row is gathered)
#pragma unroll
    for (int k = 1; k < kMaxHeavy; ++k)
        if (heavier(limit, top[k])) limit = top[k];
    rows([&](const Pick& q) {
        if (q.i == kNoRow || heavier(limit, q)) return;
        const uint32_t at = atomicAdd(&n_some, 1u);
        if (at < kGather) some[at] = q;
    });
    __syncthreads();
    const uint32_t n = n_some;
    if (n <= kGather) {
        for (uint32_t k = threadIdx.x; k < n; k += kNT) {
            const Pick q = some[k];
            uint32_t rank = 0;
#pragma unroll 4
            for (uint32_t t = 0; t < n; ++t) rank += heavier(some[t], q) ? 1u : 0u;
            if (rank < want) out[rank] = q;
        }
        if (threadIdx.x >= n && threadIdx.x < want) out[threadIdx.x] = Pick{0.0, kNoRow};
        return;
    }
    Pick last{0.0, kNoRow};
    for (uint32_t r = 0; r < want; ++r) {
        p = Pick{0.0, kNoRow};
        rows([&](const Pick& q) {
            if ((r == 0 || heavier(last, q)) && heavier(q, p)) p = q;
        });
        last = block_heaviest(p);
        if (threadIdx.x == 0) out[r] = last;
    }
}

// Candidates of one run of kHeavyRun rows: its kMaxHeavy heaviest, in order.
__global__ __launch_bounds__(kNT) void k_heavy_candidates(const double* __restrict__ m, TreeBuffers tb,
                                                          const uint32_t* __restrict__ run_sys,
                                                          Pick* __restrict__ cand)
{
    const SysScalars* sy = tb.sys + run_sys[2 * blockIdx.x];
    const uint32_t lo = sy->body_lo + run_sys[2 * blockIdx.x + 1] * kHeavyRun;
    const uint32_t hi = min(sy->body_hi, lo + kHeavyRun);
    block_top(
        kMaxHeavy,
        [&](auto f) {
#pragma unroll 8
            for (uint32_t i = lo + threadIdx.x; i < hi; i += kNT) f(pick(m[i], i));
        },
        cand + static_cast<size_t>(blockIdx.x) * kMaxHeavy);
}

// One block per system: the heaviest of its runs' candidates, ranked by row.
__global__ __launch_bounds__(kNT) void k_heavy_pick(Bodies b, TreeBuffers tb, const uint32_t* __restrict__ sys_run,
                                                    const Pick* __restrict__ cand)
{
    __shared__ Pick best[kMaxHeavy];
    const uint32_t s = blockIdx.x, r0 = sys_run[s], r1 = sys_run[s + 1];
    const uint32_t nh = tb.sys[s].n_heavy;
    if (nh == 0) return;
    // (consecutive runs go to different sets of 16 threads)
    const uint32_t first = r0 + threadIdx.x % 16 * 16 + threadIdx.x / 16;
    block_top(
        nh,
        [&](auto f) {
            for (uint32_t run = first; run < r1; run += kNT)
#pragma unroll 4
                for (int k = 0; k < kMaxHeavy; ++k) f(cand[static_cast<size_t>(run) * kMaxHeavy + k]);
        },
        best);
    __syncthreads();
    if (threadIdx.x < nh && best[threadIdx.x].i != kNoRow) {
        uint32_t rank = 0;
        for (uint32_t k = 0; k < nh; ++k) rank += best[k].i < best[threadIdx.x].i ? 1u : 0u;
        b.hrank[best[threadIdx.x].i] = static_cast<int8_t>(rank);
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
