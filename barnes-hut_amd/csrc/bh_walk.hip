// bh_walk.hip -- the plain FP64 theta-criterion walk (src/traversal.cpp:13-103).
//
// Every lane walks the compressed tree for its own body.  The tree is stored
// in walk order (pre-order, children from octant 7 down to 0, the order in
// which the reference's LIFO stack pops them), with each node's skip index
// pointing at the first node after its subtree, so a body's walk needs no
// stack: at node `cur` the lane
//   - accepts it (adds G m / r^3 * d in FP64) and continues at skip[cur],
//   - skips it (zero mass, or its own leaf) and continues at skip[cur], or
//   - opens it and continues at cur + 1.
// The lane therefore meets its accepted nodes in exactly the reference's DFS
// order and evaluates the same opening test on the same operands, so the
// accelerations are bit-identical to the reference built without FMA
// contraction.  A node stands for a unary chain of the reference's map; its
// test uses the bottom depth of the chain (see bh_tree.hip).
//
// Latency: the opening test of `cur` runs first and the record of the node
// it chooses next is fetched right away, so the fetch overlaps the FP64
// square root, division and accumulation of an accepted node instead of
// following them.  Node records are per-lane vector loads; Morton-consecutive
// lanes walk nearly the same nodes, at nearly the same time where their lead is
// limited (walk_lead), so most of them are cache hits.  The blocks are dealt
// out so that each XCD walks one contiguous eighth of the Morton order (its L2
// then holds the near field of that eighth).
// Roofline: FP64 vector (78.6 TF/s); work per body 9 flops per tested node
// + 12 per accepted node.
#include <hip/hip_runtime.h>

#include <cmath>

#include "bh_internal.hpp"

namespace bh {
namespace {

constexpr int kNT = 256;
constexpr uint32_t kXcds = 8;   // workgroup b runs on XCD b mod 8

// Full-chain bookkeeping for counters: the first depth in [top, bottom] at
// which the reference's test passes, given theta^2 r^2.
__device__ inline uint32_t first_pass_depth(const SysScalars* sy, uint32_t top, uint32_t bottom, double t2r2)
{
    uint32_t e = top;
    while (e < bottom && !(sy->side2[e] < t2r2)) ++e;
    return e;
}

// The record at walk index k; past the end (k >= T, where the lane's loop
// ends and the record is never used) the last record, so the load needs no
// branch.
__device__ inline WalkNode load_node(const WalkNode* __restrict__ walk, uint32_t k, uint32_t T)
{
    return walk[min(k, T - 1)];
}

// Block b of the grid (XCD b mod 8) -> the block of bodies it walks: XCD x
// takes blocks [x * per, (x + 1) * per) of the Morton order, per = ceil(g / 8)
// (a short last XCD range simply has fewer blocks).
__device__ inline uint32_t xcd_block(uint32_t b, uint32_t g)
{
    const uint32_t per = (g + kXcds - 1) / kXcds;
    const uint32_t x = b % kXcds, k = b / kXcds;
    return x * per + k;
}

// set bits of m below this lane
__device__ inline uint32_t rank_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

__device__ inline uint64_t read_lane(uint64_t v, int from)
{
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), from));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), from));
    return static_cast<uint64_t>(hi) << 32 | lo;
}

struct Decision {
    double dx, dy, dz, r2, t2r2;
    bool live, is_self, accept, open;
};

// The decision at a node (src/traversal.cpp:67-77): zero-mass nodes and the
// body's own leaf are skipped, a leaf is always accepted, a cell when side^2 <
// theta^2 r^2.  (A leaf is accepted always except by its own bodies: their
// leaf's side^2 is +inf unless its chain starts above depth 21, so `pass` is
// the reference's self-chain test.  Bitwise, so the decision is a few mask
// operations and no branch.)
__device__ inline Decision decide(const WalkNode& nd, double px, double py, double pz, bool is_self,
                                  const WalkParams& p)
{
    Decision d;
    d.dx = nd.x - px;
    d.dy = nd.y - py;
    d.dz = nd.z - pz;
    d.r2 = d.dx * d.dx + d.dy * d.dy + d.dz * d.dz + p.soft2;
    d.t2r2 = p.theta2 * d.r2;
    d.live = nd.m != 0.0;
    d.is_self = is_self;
    const bool pass = nd.side2 < d.t2r2;
    const bool leaf = (nd.meta & kMetaLeaf) != 0u;
    d.accept = d.live & (pass | (leaf & !is_self));
    d.open = d.live & !d.accept & !is_self;
    return d;
}

// G m / r^3.  inv_sqrt_in_range gives the bits of 1.0 / sqrt(r2) where it takes
// r2; a wave with a lane whose r2 it does not takes the library path.
__device__ inline double pull(double r2, double m, double G)
{
    const double invR = __ballot(!inv_sqrt_takes(r2)) == 0ull ? inv_sqrt_in_range(r2) : 1.0 / sqrt(r2);
    const double invR3 = invR * invR * invR;
    return G * m * invR3;
}

// the smallest v of the wavefront (all lanes active), in a scalar
template <int kCtrl, int kRows>
__device__ inline uint32_t dpp_min(uint32_t v)
{
    return min(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), kCtrl, kRows,
                                                                  0xf, false)));
}

__device__ inline uint32_t wave_min(uint32_t v)
{
    v = dpp_min<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v = dpp_min<0x112, 0xf>(v);
    v = dpp_min<0x114, 0xf>(v);
    v = dpp_min<0x118, 0xf>(v);
    v = dpp_min<0x142, 0xa>(v);   // row_bcast 15, 31
    v = dpp_min<0x143, 0xc>(v);
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// Visits between two looks at where the last lane is (kLead; 4 and 16 measured
// the same).
constexpr int kVisits = 8;

template <bool kCount, bool kLead>
__global__ __launch_bounds__(kNT) void k_walk_plain(Bodies b, size_t n, uint32_t grid_blocks,
                                                    const WalkNode* __restrict__ walk,
                                                    const uint32_t* __restrict__ self_w,
                                                    const StepScalars* __restrict__ sc,
                                                    const SysScalars* __restrict__ sy, WalkParams p, uint32_t lead,
                                                    int64_t* __restrict__ cnt_accept, int64_t* __restrict__ cnt_open,
                                                    int64_t* __restrict__ cnt_test)
{
    const uint32_t vb = xcd_block(blockIdx.x, grid_blocks);
    const size_t i = static_cast<size_t>(vb) * kNT + threadIdx.x;
    // M + B <= 2n - 1 by construction; the clamp keeps a corrupted count in bounds
    const uint32_t T = min(sc->n_nodes, static_cast<uint32_t>(2 * n));
    if (T * sizeof(WalkNode) <= kWarmBytes) warm_l2(walk, T * sizeof(WalkNode));
    // (a lane without a body has arrived; it takes part in the wavefront's minima)
    const size_t ib = min(i, n - 1);
    const double px = b.px[ib];
    const double py = b.py[ib];
    const double pz = b.pz[ib];
    const uint32_t self = self_w[ib];
    double ax = 0.0, ay = 0.0, az = 0.0;
    int64_t na = 0, no = 0, nt = 0;
    uint32_t cur = i < n ? 0u : T;
    WalkNode nd = load_node(walk, 0, T);
    const auto visit = [&]() {
        // the decision first
        const Decision d = decide(nd, px, py, pz, cur == self, p);
        // then the fetch of the next record, whose latency the FP64
        // arithmetic of the accepted node covers; a subtree's skip index
        // always lies beyond it, and max() keeps the walk moving forward even
        // for a corrupted record
        const uint32_t next = d.open ? cur + 1 : max(nd.skip, cur + 1);
        const WalkNode nn = load_node(walk, next, T);
        if (d.accept) {
            const double s = pull(d.r2, nd.m, p.G);
            ax += s * d.dx;
            ay += s * d.dy;
            az += s * d.dz;
        }
        if (kCount && d.live) {
            ++nt;
            const uint32_t top = (nd.meta >> kMetaTopShift) & 31u;
            const uint32_t bottom = nd.meta & kMetaDepthMask;
            if (d.accept) {
                ++na;
                // the reference opens the chain cells above the first passing depth
                const bool leaf = (nd.meta & kMetaLeaf) != 0u;
                const uint32_t last = leaf ? (d.is_self ? kMaxDepth - 1 : kMaxDepth) : bottom;
                no += first_pass_depth(sy, top, last, d.t2r2) - top;
            } else if (d.is_self) {
                no += kMaxDepth - top;
            } else {
                no += bottom - top + 1;
            }
        }
        cur = next;
        nd = nn;
    };
    if constexpr (kLead) {
        for (;;) {
            const uint32_t last = wave_min(cur);
            if (last >= T) break;
            const uint32_t ahead = lead < T - last ? last + lead : T - 1;
            for (int r = 0; r < kVisits; ++r)
                if (cur <= ahead) visit();
        }
    } else {
        while (cur < T) visit();
    }
    if (i >= n) return;
    b.ax[i] = ax;
    b.ay[i] = ay;
    b.az[i] = az;
    if (p.kick) {
        // src/main.cpp:278-280: v += 0.5 * dt * a
        b.vx[i] = b.vx[i] + p.half_dt * ax;
        b.vy[i] = b.vy[i] + p.half_dt * ay;
        b.vz[i] = b.vz[i] + p.half_dt * az;
    }
    if (kCount) {
        cnt_accept[i] = na;
        cnt_open[i] = no;
        cnt_test[i] = nt;
    }
}

// ----------------------------------------------------- a small system's walk
// One wavefront walks one body.  The per-lane walk above is one chain of
// dependent visits per body, and a small system has too few bodies to fill the
// chip with such chains; here the nodes still to be visited lie on a stack in
// LDS, up to 128 are visited at once, and a visit pushes the first and the
// middle child of an opened node and the next sibling of its chain.  The
// visits come in no order, so an accepted node is also a bit in a bitmap over
// the walk indices: the bits below it are its rank in the reference's order.
// The contributions are then evaluated 64 at a time in that order, and three
// lanes add them up one by one, while the next 64 records are on their way: the
// bits of the per-lane walk.
// LDS: 2 n bits for the bitmap; the stack, whose place the counts before each
// word of the bitmap take, and then the contributions; and the accepted nodes
// as they were found, whose place the ordered ones take.  More than kFound are
// read off the bitmap in pieces instead.  A full stack, or more visits than
// the tree has nodes, sends the body to the walk by one lane (walk_alone).
// Walks of a belt, theta 1.05, per lane and by wavefronts: 3,000 bodies 0.121 and
// 0.028 ms, 8,000 0.188 and 0.072, 20,480 0.277 and 0.204, the last bound by
// vector instructions and by the latency of a wavefront's rounds (16 wavefronts a
// CU, by their LDS).  Where the lists are short the lanes are faster: short_lists.
constexpr uint32_t kStack = 1024;       // (950 the deepest seen with no limit, at theta 0.1)
constexpr uint32_t kFound = 1536;
constexpr uint32_t kWaves = 4;          // bodies of a block, independent of each other
constexpr uint32_t kConRow = 66;        // contributions of one component: 64 and a pad for the banks

struct alignas(16) WaveLds {
    union {
        uint16_t stack[kStack];
        uint16_t before[2 * kWaveMax / 64];
        double con[3][kConRow];
    };
    uint16_t list[kFound];
};

template <int kCtrl, int kRows>
__device__ inline uint32_t dpp_add(uint32_t v)
{
    return v + static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, kRows, 0xf, false));
}

__device__ inline uint32_t wave_scan(uint32_t v)   // inclusive prefix sum
{
    v = dpp_add<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);   // row_bcast 15, 31
    return dpp_add<0x143, 0xc>(v);
}

__device__ inline void store_acc(const Bodies& b, size_t i, uint32_t c, double a, const WalkParams& p)
{
    (c == 0 ? b.ax : c == 1 ? b.ay : b.az)[i] = a;
    if (!p.kick) return;
    double* v = (c == 0 ? b.vx : c == 1 ? b.vy : b.vz) + i;
    *v = *v + p.half_dt * a;   // src/main.cpp:278-280
}

struct Vec3 {
    double x, y, z;
};

__device__ inline Vec3 contribution(const WalkNode& nd, double px, double py, double pz, const WalkParams& p)
{
    const double dx = nd.x - px;
    const double dy = nd.y - py;
    const double dz = nd.z - pz;
    const double r2 = dx * dx + dy * dy + dz * dz + p.soft2;
    const double s = pull(r2, nd.m, p.G);
    return {s * dx, s * dy, s * dz};
}

__device__ inline void store_acc(const Bodies& b, size_t i, const Vec3& a, const WalkParams& p)
{
    store_acc(b, i, 0, a.x, p);
    store_acc(b, i, 1, a.y, p);
    store_acc(b, i, 2, a.z, p);
}

// One body's walk by one lane; the fetch of the next record comes before the
// arithmetic of an accepted one.
__device__ inline Vec3 walk_alone(const WalkNode* __restrict__ walk, uint32_t T, double px, double py, double pz,
                                  uint32_t self, const WalkParams& p)
{
    Vec3 a{0.0, 0.0, 0.0};
    WalkNode nd = load_node(walk, 0, T);
    for (uint32_t cur = 0; cur < T;) {
        const Decision d = decide(nd, px, py, pz, cur == self, p);
        const uint32_t next = d.open ? cur + 1 : max(nd.skip, cur + 1);
        const WalkNode nn = load_node(walk, next, T);
        if (d.accept) {
            const double s = pull(d.r2, nd.m, p.G);
            a.x += s * d.dx;
            a.y += s * d.dy;
            a.z += s * d.dz;
        }
        cur = next;
        nd = nn;
    }
    return a;
}

// Whether the per-lane walk is the faster one, by the tests of a mean body V:
// 32 V < n - kWaveFew.  A wavefront's time for a body hardly depends on its
// list, a lane's is proportional to it.  (n and theta alone do not tell: the
// same limits for all had Kuiper belts of 20,480 bodies walked 1.4 times as long
// as per lane, cubes 1.7 times, at the theta at which belts gain.)  Walks in us
// per lane and by wavefronts (belt, Kuiper belt, cube; V in brackets): 8,192
// bodies theta 1.05 190, 73 (677), 90, 54 (212), 44, 36 (78); 12,288 theta 1.05
// 218, 116 (786), 81, 86 (226), 48, 55 (84); 20,480 theta 1.05 285, 200 (894),
// 100, 139 (279), 53, 91 (90), theta 0.5 744, 664 (2,990), 315, 253 (1,121), 171,
// 143 (532).  Over seven shapes, 5,000 to 20,480 bodies and theta 0.3 to 3 the
// choice is within 5% of the better walk in 356 of 378 cases, and up to theta 1.2
// in 246 of 252; 1.26 the worst of those (a cube of 8,192 bodies, 44 us for 35).
__device__ inline bool short_lists(const StepScalars* sc, size_t n)
{
    uint32_t tests = 0;
#pragma unroll
    for (uint32_t x = 0; x < kXcds; ++x) tests += sc->queue[x][0];
    static_assert(kListSamples == 16, "the tests of the samples are 16 V");
    return 2 * tests < n - kWaveFew;
}

// Orders this wavefront's LDS accesses for its lanes (the LDS serves one
// wavefront's instructions in order, so nothing is waited for).
__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(64 * kWaves) void k_walk_wave(Bodies b, size_t n, uint32_t grid_blocks,
                                                           const WalkNode* __restrict__ walk,
                                                           const uint32_t* __restrict__ self_w,
                                                           const StepScalars* __restrict__ sc, WalkParams p,
                                                           uint32_t words)
{
    extern __shared__ unsigned long long all_bits[];
    __shared__ WaveLds ls[kWaves];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    unsigned long long* const bits = all_bits + wave * words;
    WaveLds& l = ls[wave];
    const uint32_t T = min(sc->n_nodes, static_cast<uint32_t>(2 * n));
    if (counts_lists(n) && short_lists(sc, n)) {
        // per lane, as k_walk_plain does it
        const uint32_t g = static_cast<uint32_t>((n + 64 * kWaves - 1) / (64 * kWaves)), used = (g + kXcds - 1) / kXcds * kXcds;
        if (blockIdx.x >= used) return;
        warm_l2<64 * kWaves>(walk, T * sizeof(WalkNode), used);
        const size_t i = static_cast<size_t>(xcd_block(blockIdx.x, g)) * (64 * kWaves) + threadIdx.x;
        if (i < n) store_acc(b, i, walk_alone(walk, T, b.px[i], b.py[i], b.pz[i], self_w[i], p), p);
        return;
    }
    warm_l2<64 * kWaves>(walk, T * sizeof(WalkNode));
    const size_t i = static_cast<size_t>(xcd_block(blockIdx.x, grid_blocks)) * kWaves + wave;
    if (i >= n || T == 0) return;
    const double px = b.px[i];
    const double py = b.py[i];
    const double pz = b.pz[i];
    const uint32_t self = self_w[i];
    for (uint32_t k = lane; k < words; k += 64) bits[k] = 0;
    if (lane == 0) l.stack[0] = 0;
    wave_sync();

    uint32_t size = 1, visits = 0, total = 0;   // total: accepted nodes
    // the visit of node k by the lanes with act: at most three pushes each
    const auto visit = [&](bool act, uint32_t k, const WalkNode& nd) {
        const Decision d = decide(nd, px, py, pz, k == self, p);
        const bool take = act & d.accept;
        const uint64_t mt = __ballot(take);
        const uint32_t at = total + rank_below(mt);
        if (take) atomicOr(bits + (k >> 6), 1ull << (k & 63u));
        if (take & (at < kFound)) l.list[at] = static_cast<uint16_t>(k);
        total += static_cast<uint32_t>(__popcll(mt));
        const uint32_t mid = nd.meta >> kMetaMidShift & 0xffffu;
        const bool more = act & ((nd.meta & kMetaMore) != 0u) & (nd.skip > k) & (nd.skip < T);
        const bool open = act & d.open & (k + 1 < T);
        const bool open2 = open & (mid > k) & (mid < T);
        const uint64_t mm = __ballot(more), mo = __ballot(open), m2 = __ballot(open2);
        const uint32_t s2 = size + static_cast<uint32_t>(__popcll(mm));
        const uint32_t s3 = s2 + static_cast<uint32_t>(__popcll(m2));
        const uint32_t s4 = s3 + static_cast<uint32_t>(__popcll(mo));
        if (more) l.stack[size + rank_below(mm)] = static_cast<uint16_t>(nd.skip);
        if (open2) l.stack[s2 + rank_below(m2)] = static_cast<uint16_t>(mid);
        if (open) l.stack[s3 + rank_below(mo)] = static_cast<uint16_t>(k + 1);
        size = s4;
    };
    bool ok = true;
    while (ok && size > 0) {
        // near a full stack fewer are visited at once: t leave it, at most 3 t come
        const uint32_t t = min(min(size, 128u), (kStack - size) / 2);
        if (t == 0) {
            ok = false;
            break;
        }
        size -= t;
        visits += t;
        const bool a0 = lane < t, a1 = lane + 64 < t;
        const uint32_t k0 = l.stack[size + (a0 ? lane : 0u)];
        const WalkNode n0 = load_node(walk, k0, T);
        if (t > 64) {
            const uint32_t k1 = l.stack[size + (a1 ? lane + 64 : 0u)];
            const WalkNode n1 = load_node(walk, k1, T);
            wave_sync();
            visit(true, k0, n0);
            visit(a1, k1, n1);
        } else {
            wave_sync();
            visit(a0, k0, n0);
        }
        if (visits > T) ok = false;
        wave_sync();
    }
    wave_sync();

    if (!ok) {
        if (lane == 0) store_acc(b, i, walk_alone(walk, T, px, py, pz, self, p), p);
        return;
    }

    uint32_t cnt = 0;                 // ordered indices in l.list
    uint32_t next = 0;                // where they are read off: the bitmap's next 64 words,
    uint64_t word = 0, left = 0;      // the lane's of the last 64, those not yet read
    if (total <= kFound) {
        uint32_t f[kFound / 64];
#pragma unroll
        for (uint32_t q = 0; q < kFound / 64; ++q)
            if (q * 64 < total) f[q] = l.list[min(q * 64 + lane, total - 1)];
        for (uint32_t w0 = 0; w0 < words; w0 += 64) {
            const uint32_t w = w0 + lane;
            const uint32_t c = w < words ? static_cast<uint32_t>(__popcll(bits[w])) : 0u;
            const uint32_t inc = wave_scan(c);
            if (w < words) l.before[w] = static_cast<uint16_t>(cnt + inc - c);
            cnt += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(inc), 63));
        }
        wave_sync();
        // (the nodes visited are distinct, and so are their ranks; the lanes
        // past the end write the last one's again)
        cnt = min(cnt, kFound);
#pragma unroll
        for (uint32_t q = 0; q < kFound / 64; ++q)
            if (q * 64 < total) {
                const uint64_t below = bits[f[q] >> 6] & ((1ull << (f[q] & 63u)) - 1ull);
                const uint32_t r = l.before[f[q] >> 6] + static_cast<uint32_t>(__popcll(below));
                l.list[min(r, kFound - 1)] = static_cast<uint16_t>(f[q]);
            }
        next = words;
    }
    double acc = 0.0;   // lane c: component c
    const uint32_t row = min(lane, 2u);
    const auto put = [&](uint32_t j, const Vec3& c) {
        // (a sum that starts at 0.0 is never -0.0, so adding 0.0 keeps its bits)
        const bool in = j + lane < cnt;
        l.con[0][lane] = in ? c.x : 0.0;
        l.con[1][lane] = in ? c.y : 0.0;
        l.con[2][lane] = in ? c.z : 0.0;
    };
    const auto add_up = [&]() {
        const double2* v = reinterpret_cast<const double2*>(l.con[row]);
#pragma unroll 1
        for (uint32_t g = 0; g < 32; g += 8) {   // (all of it at once would take 128 registers)
            double2 c[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) c[u] = v[g + u];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                acc += c[u].x;
                acc += c[u].y;
            }
        }
    };
    do {
        if (left != 0 || next < words) {
            cnt = 0;
            while (cnt <= kFound - 64) {
                if (left == 0) {
                    if (next >= words) break;
                    word = next + lane < words ? bits[next + lane] : 0;
                    left = __ballot(word != 0);
                    next += 64;
                    continue;
                }
                const int from = __ffsll(static_cast<unsigned long long>(left)) - 1;
                left &= left - 1;
                const uint64_t w = read_lane(word, from);
                const uint32_t k0 = (next - 64 + static_cast<uint32_t>(from)) * 64;
                if (w >> lane & 1) l.list[cnt + rank_below(w)] = static_cast<uint16_t>(k0 + lane);
                cnt += static_cast<uint32_t>(__popcll(w));
            }
        }
        wave_sync();
        if (cnt == 0) continue;
        put(0, contribution(load_node(walk, l.list[min(lane, cnt - 1)], T), px, py, pz, p));
        wave_sync();
        for (uint32_t j = 64; j < cnt; j += 64) {
            const WalkNode nd = load_node(walk, l.list[min(j + lane, cnt - 1)], T);
            add_up();
            wave_sync();
            put(j, contribution(nd, px, py, pz, p));
            wave_sync();
        }
        add_up();
        wave_sync();
    } while (left != 0 || next < words);
    if (lane < 3) store_acc(b, i, lane, acc, p);
}

// How many walk indices a lane may be ahead of its wavefront's last one (0: no
// limit).  The lanes of a wavefront drift apart, and then every lane's record
// is a line of its own: 44 lines a visit at 300k bodies, one L1 lookup each for
// each of the record's three loads, and at one lookup a clock these are what
// bounds a full chip (vector instructions 37% busy).  Lanes that wait for the
// last one make the visits share lines; their steps are more (simulated at
// 300k, theta 1.05, limit 5,000: 23 lines a visit, 19% more steps), which a chip
// with few wavefronts pays for.  Walks in ms, no limit and 30,000 / 10,000 /
// 4,000 / 1,000: belt 50,000 theta 1.05 0.48, 0.52 / 0.56 / 0.68 / 0.83; 130,000
// 0.94, 0.89 / 1.03 / 1.12 / 1.25; 300k 2.12, 2.06 / 2.04 / 2.08 / 2.20, theta
// 0.5 11.6, 11.0 / 10.7 / 10.4 / 10.1; Trojan 300k theta 0.7 5.4, 5.1 / 4.9 /
// 4.6 / 4.3; Kuiper 300k theta 0.7 1.35, 1.24 / 1.20 / 1.20 / 1.28; Trojan 1M
// 7.8, 6.7 / 6.1 / 5.9 / 5.8.  With the rule against no limit, belt / Trojan /
// Kuiper: 100k theta 0.5 0.96 / 0.96 / 1.01, 1.05 0.98 / 0.96 / 1.06; 130k theta
// 0.5 0.92 / 0.96 / 0.98, 1.05 0.94 / 0.98 / 0.99; 300k theta 1.05 0.94 / 0.91 /
// 0.94, 2 0.93 / 0.91 / 1.10; 1M theta 1.05 0.81 / 0.79 / 0.91.  Above theta 1.2
// it lost below 160k: 100k theta 1.5 0.97 / 1.06 / 1.04, 2 1.12 / 1.09 / 1.08,
// 130k 1.5 1.04 / 1.01 / 1.03, 2 1.06 / 1.10 / 1.08.
uint32_t walk_lead(size_t n, double theta2)
{
    if (n < 100000) return 0u;
    if (n < 160000) return theta2 > 1.44 ? 0u : 30000u;
    return theta2 < 0.64 ? 4000u : 10000u;
}

}  // namespace

void launch_walk_plain(const Bodies& b, size_t n, const TreeBuffers& tb, const WalkParams& p,
                       int64_t* cnt_accept, int64_t* cnt_open, int64_t* cnt_test, hipStream_t s)
{
    const uint32_t g = static_cast<uint32_t>((n + kNT - 1) / kNT);
    if (g == 0) return;
    // the XCD-contiguous mapping covers blocks [0, 8 * ceil(g / 8)); blocks
    // mapped past g have no bodies, but take their part in the L2 sweep, whose
    // slices count every block of the grid
    const uint32_t grid = ((g + kXcds - 1) / kXcds) * kXcds;
    const uint32_t lead = walk_lead(n, p.theta2);
    if (cnt_accept && cnt_open && cnt_test)
        k_walk_plain<true, false><<<grid, kNT, 0, s>>>(b, n, g, tb.walk, tb.self_w, tb.sc, tb.sys, p, 0u, cnt_accept, cnt_open,
                                                cnt_test);
    else if (n <= kWaveMax) {
        const uint32_t words = static_cast<uint32_t>((2 * n + 63) / 64);
        const uint32_t gw = static_cast<uint32_t>((n + kWaves - 1) / kWaves);
        k_walk_wave<<<(gw + kXcds - 1) / kXcds * kXcds, 64 * kWaves, kWaves * words * sizeof(uint64_t), s>>>(
            b, n, gw, tb.walk, tb.self_w, tb.sc, p, words);
    } else if (lead != 0u)
        k_walk_plain<false, true><<<grid, kNT, 0, s>>>(b, n, g, tb.walk, tb.self_w, tb.sc, tb.sys, p, lead, nullptr, nullptr,
                                                 nullptr);
    else
        k_walk_plain<false, false><<<grid, kNT, 0, s>>>(b, n, g, tb.walk, tb.self_w, tb.sc, tb.sys, p, 0u, nullptr, nullptr,
                                                 nullptr);
}

}  // namespace bh
