// bh_direct.hip -- FP64 direct-sum accelerations for sample bodies, the
// error reference for every walk form.  A sample sees the bodies of its own
// system only (systems are independent).  A block of 256 threads takes R
// samples; each thread runs one compensated sum per sample over a strided
// share of the bodies, and a sample's 256 compensated partials are combined in
// thread order, so the result depends neither on R nor on the other samples.
//
// Bound by the FP64 units: about 58 wave instructions a pair (17 of them the
// reciprocal square root without its range handling, 21 the three compensated
// additions), issued at 80% of the rate at the clock the card holds (2.05
// GHz).  R samples share the loads of a body and the range check, and their
// square roots overlap; one sample a block streamed the bodies from L2 at 10
// TB/s.  4,096 samples of 300,149 bodies: 3.70 -> 2.89 ms; 512: 0.86 -> 0.57.
#include <hip/hip_runtime.h>

#include <cmath>

#include "bh_internal.hpp"

namespace bh {
namespace {

constexpr int kNT = 256;

// Samples of one system only share a pass (the systems' ranges differ);
// samples past m repeat the last one and are not written.
template <int R>
__global__ __launch_bounds__(kNT) void k_direct_sum(Bodies b, TreeBuffers tb, const int64_t* __restrict__ idx,
                                                    int64_t m, double G, double soft2, double* __restrict__ acc3)
{
    __shared__ double part[3][kNT];
    const int64_t first = static_cast<int64_t>(blockIdx.x) * R;
    int64_t i[R];
    double px[R], py[R], pz[R];
    ExactSum ax[R], ay[R], az[R];
    size_t j0[R], j1[R];
    bool one_system = true;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        i[r] = idx[first + r < m ? first + r : m - 1];
        px[r] = b.px[i[r]];
        py[r] = b.py[i[r]];
        pz[r] = b.pz[i[r]];
        const SysScalars* sy = tb.sys + tb.bsys[i[r]];
        j0[r] = sy->body_lo;
        j1[r] = sy->body_hi;
        one_system &= j0[r] == j0[0];
    }
    // body j's terms of the samples [r0, r1); a sample skips itself and
    // co-located bodies.  One range check serves every sample, so that their
    // square roots overlap.
    auto terms = [&](int r0, int r1, size_t j, double x, double y, double z, double gm) {
        double dx[R], dy[R], dz[R], q[R];
        bool pair[R], fast = true;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r < r0 || r >= r1) continue;
            dx[r] = x - px[r];
            dy[r] = y - py[r];
            dz[r] = z - pz[r];
            q[r] = dx[r] * dx[r] + dy[r] * dy[r] + dz[r] * dz[r] + soft2;
            pair[r] = static_cast<int64_t>(j) != i[r] && q[r] > 0.0;
            fast &= inv_sqrt_takes(q[r]) | !pair[r];
        }
        double invR[R];
        if (__all(fast)) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r >= r0 && r < r1) invR[r] = inv_sqrt_in_range(q[r]);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r >= r0 && r < r1) invR[r] = 1.0 / sqrt(q[r]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r < r0 || r >= r1) continue;
            if (pair[r]) {
                const double f = gm * (invR[r] * invR[r] * invR[r]);
                ax[r].add(f * dx[r]);
                ay[r].add(f * dy[r]);
                az[r].add(f * dz[r]);
            }
        }
    };
    if (one_system) {
        for (size_t j = j0[0] + threadIdx.x; j < j1[0]; j += kNT)
            terms(0, R, j, b.px[j], b.py[j], b.pz[j], G * b.m[j]);
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
            for (size_t j = j0[r] + threadIdx.x; j < j1[r]; j += kNT)
                terms(r, r + 1, j, b.px[j], b.py[j], b.pz[j], G * b.m[j]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        part[0][threadIdx.x] = ax[r].value();
        part[1][threadIdx.x] = ay[r].value();
        part[2][threadIdx.x] = az[r].value();
        __syncthreads();
        if (threadIdx.x < 3 && first + r < m) {
            ExactSum t;
            for (int k = 0; k < kNT; ++k) t.add(part[threadIdx.x][k]);
            acc3[3 * (first + r) + threadIdx.x] = t.value();
        }
        __syncthreads();
    }
}

}  // namespace

void launch_direct_sum(const Bodies& b, const TreeBuffers& tb, const int64_t* idx, size_t m, double G, double soft2,
                       double* acc3, hipStream_t s)
{
    if (m == 0) return;
    const int64_t mm = static_cast<int64_t>(m);
    // several samples a block while that leaves the 256 CUs blocks to take
    if (m >= 4096) k_direct_sum<4><<<static_cast<unsigned>((m + 3) / 4), kNT, 0, s>>>(b, tb, idx, mm, G, soft2, acc3);
    else if (m >= 1024) k_direct_sum<2><<<static_cast<unsigned>((m + 1) / 2), kNT, 0, s>>>(b, tb, idx, mm, G, soft2, acc3);
    else k_direct_sum<1><<<static_cast<unsigned>(m), kNT, 0, s>>>(b, tb, idx, mm, G, soft2, acc3);
}

}  // namespace bh
