// bh_mixed.hip -- the precision form of the walk: FP32 on group-relative
// offsets with compensated accumulation, FP64 for the heavy bodies.
//
// Walk groups.  Bodies are cut into groups of at most 64 Morton-consecutive
// bodies that follow the tree: a cell with <= 64 bodies whose parent holds
// more is a bucket; consecutive sibling buckets are packed while they fit in
// 64; a leaf with more than 64 co-keyed bodies is split.  The tree is walked
// once per group: by one wavefront, or by the four of a block for a group that
// would end late (share_limit), with the same bits.
//
// Opening test per group (the extent test): a node is accepted when
// b^2 < theta^2 * D^2, with b the distance from the node's centre of mass to
// the farthest corner of the bounding box of its light bodies (the node's true
// extent, <= the cell diagonal) and D the FP64 distance from that centre of mass to the group's
// bounding box.  Every body of the group is at least D away, so each body
// sees the node inside a cone of half-angle ~theta, the same accuracy class
// as the reference's per-body test (src/traversal.cpp:78), but measured on
// the bodies actually present instead of the cubic cell.  The result of a
// group depends only on the group, never on which worker walks it or when:
// every schedule gives identical bits.  For theta > 0.8 a second, relative
// test guards the nodes with b > 0.8 D, where the monopole error bound grows
// without limit as b/D -> 1: such a node is accepted only if its quadrupole
// scale G Q / D^4 (Q = sum m |x - com|^2 of its light bodies) is at most
// alpha times the smallest heavy-body acceleration of the group.
//
// Traversal keeps a stack of node ranges in LDS (children of a node occupy
// consecutive slots); each round pops up to 64 ranges, one per lane, and the
// lanes test the nodes of their range in FP64.  Accepted nodes and the bodies
// of reached leaves go into an LDS interaction list as FP32 (x - c, y - c,
// z - c, G m) with c the group centre (FP64), so the offsets keep FP32
// precision near the group.  A full list is cut into shares, one for each of
// up to 256 virtual lanes (share and body) whatever the group's size, and
// evaluated in FP32 FMA over blocks of 32 entries, each block sum added into a
// Kahan-compensated FP32 accumulator.  A group's own bodies appear in the
// list with offsets bit-identical to the lane's own, so the self term has
// dx = dy = dz = 0 and adds +0 (r^2 starts from a small positive floor).
//
// Heavy bodies (the central mass and planets: the heaviest bodies, up to 16)
// are not in the light moments; every light body adds them by an FP64 direct
// sum (the ranks k = q mod 4 into partial q, in rank order, then the four
// partials), and the heavy bodies themselves get an FP64 direct sum over all
// bodies (heavy_item, k_heavy_final).  The sum of the two parts is FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "bh_internal.hpp"

namespace bh {
namespace {

constexpr int kNT = 256;
constexpr int kWaves = kNT / 64;
// kShare = 0.6.  Walk, ms (cost order, key order), kShare 0.2 / 0.6 / 1.0 /
// no sharing: 50k bodies 0.128, 0.150 / 0.128, 0.147 / 0.125, 0.149 / 0.197,
// 0.200; 200k key order 0.436 / 0.330 / 0.424 / 0.416; 300k 0.475, 0.520 /
// 0.437, 0.493 / 0.440, 0.490 / 0.428, 0.486.  A shared group's round costs a
// third more wave time than a lone wavefront's (its barriers, and four
// wavefronts working out the same ranges), so sharing pays only for groups
// that would end late, and the limit grows with the groups per wave.
constexpr uint32_t kShareNum = 3, kShareDen = 5;
constexpr int kListCap = 256;
constexpr int kListPad = 64;    // zero entries past a flushed list (share_len)
constexpr int kStackCap = 1024;
// One round pushes at most 8 ranges per popped range, and a single-range round
// (pure depth first) grows the stack by at most 7 per level: P ranges may be
// popped while 7 P more fit below the room of one descent.  (Popping 64 or,
// near the limit, one at a time: a group of four far-apart planets, which opens
// 33,000 nodes of a 300k belt, walked 5.7 nodes a round; the belt's walk 3.78 ->
// 0.52 ms with this rule.  A 64-system belt ensemble of 3.8M bodies 18.7 ->
// 5.6 ms.  Groups that do not fill their stack
// are walked as before.)
// narrow: 64 or one at a time.  The work of a group, the target of the learned
// form's training, depends on where the list is flushed and so on the order of
// its entries: a training walk counts it in the narrow order, by a second pass
// without forces over the groups for which the two differ.
constexpr uint32_t kStackRoom = kStackCap - 8 * 22;
constexpr uint32_t kNarrowRoom = kStackRoom - 7 * 64;   // both rules are the same up to here
__device__ inline uint32_t pop_count(uint32_t sp, bool narrow)
{
    if (narrow) return sp <= kNarrowRoom ? min(sp, 64u) : 1u;
    const uint32_t fit = sp < kStackRoom ? (kStackRoom - sp) / 7u : 0u;
    return min(min(sp, 64u), max(fit, 1u));
}
constexpr uint32_t kNone = 0xffffffffu;
// b/D at or below 0.8 keeps the monopole error bound of an accepted node
// (which grows like (b/D)^2 / (1 - b/D)^2) small; above it, up to theta, the
// relative quadrupole test decides as well
constexpr double kSafe2 = 0.64;

// Cell occupancy by depth, per system: sys[s].dcount[d] = number of
// boundaries u[j] | u[j+1] inside system s that split at depth d, so depth d
// holds 1 + sum_{e < d} dcount[e] non-empty cells of s.  With one system each
// wavefront counts 64 boundaries per round with one ballot per depth; with
// several, LDS counters per (system, depth).  Blocks add their counts into
// dcount, which sys_extents (block 0 of k_slots) reads and clears.
// Histogram blocks: one per 4,096 bodies, at least 128 and at most 2,048, so
// each wavefront takes about 16 rounds of 64 boundaries (with 128 blocks at
// 4.1M bodies each took 126 rounds of dependent loads: 261 us).
inline unsigned hist_blocks(size_t n)
{
    return static_cast<unsigned>(std::min<size_t>(2048, std::max<size_t>(128, n / 4096)));
}

__device__ inline void split_hist(const TreeBuffers& tb, uint32_t hist_grid)
{
    __shared__ uint32_t h[kMaxSystems][kMaxDepth + 1];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t M = tb.sc->n_leaves;
    const uint32_t rows = tb.n_sys;
    for (uint32_t k = threadIdx.x; k < rows * (kMaxDepth + 1); k += kNT) (&h[0][0])[k] = 0;
    __syncthreads();
    const uint32_t stride = hist_grid * kNT;
    if (rows == 1) {
        uint32_t cnt[kMaxDepth + 1];
#pragma unroll
        for (int d = 0; d <= kMaxDepth; ++d) cnt[d] = 0;
        for (uint32_t j0 = blockIdx.x * kNT + w * 64; j0 + 1 < M; j0 += stride) {
            const uint32_t j = j0 + static_cast<uint32_t>(lane);
            const int d = (j + 1 < M) ? static_cast<int>(tb.delta[j]) : -1;
#pragma unroll
            for (int e = 0; e <= kMaxDepth; ++e) cnt[e] += static_cast<uint32_t>(__popcll(__ballot(d == e)));
        }
        if (lane == 0)
            for (int d = 0; d <= kMaxDepth; ++d) atomicAdd(&h[0][d], cnt[d]);
    } else {
        // a wavefront whose 64 boundaries all lie in one system (nearly all of
        // them: systems hold thousands of leaves) counts them with one ballot
        // per depth, like the single-system case; others count lane by lane
        for (uint32_t j0 = blockIdx.x * kNT + w * 64; j0 + 1 < M; j0 += stride) {
            const uint32_t j = j0 + static_cast<uint32_t>(lane);
            const bool in = j + 1 < M;
            const int d = in ? static_cast<int>(tb.delta[j]) : -1;   // kNoSplit is never a depth
            const uint32_t sy = in ? static_cast<uint32_t>(tb.bsys[tb.leaf_first[j]]) : 0u;
            const uint32_t s0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(sy)));
            if (__all(!in || sy == s0)) {
#pragma unroll
                for (int e = 0; e <= kMaxDepth; ++e) {
                    const uint32_t c = static_cast<uint32_t>(__popcll(__ballot(d == e)));
                    if (lane == 0 && c) atomicAdd(&h[s0][e], c);
                }
            } else if (in && d != kNoSplit) {
                atomicAdd(&h[sy][d], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < rows * (kMaxDepth + 1); k += kNT) {
        const uint32_t v = (&h[0][0])[k];
        if (v) atomicAdd(&tb.sys[k / (kMaxDepth + 1)].dcount[k % (kMaxDepth + 1)], v);
    }
}

// number of children of every branching node (into base, scanned next)
__device__ inline uint32_t child_count(const TreeBuffers& tb, size_t bi)
{
    uint32_t c = 0;
    if (bi < tb.sc->n_branch) {
        const int32_t* ch = tb.child + 8 * bi;
#pragma unroll
        for (int k = 0; k < 8; ++k) c += ch[k] >= 0 ? 1u : 0u;
    }
    return c;
}

// The first hist_grid blocks count the split depths; every block over the
// branching nodes also leaves the block sum of their child counts (k_slots
// scans them).
__global__ __launch_bounds__(kNT) void k_split_hist(size_t n, TreeBuffers tb, uint32_t hist_grid)
{
    const size_t bi = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    const uint32_t cc = bi < n ? child_count(tb, bi) : 0u;
    if (blockIdx.x < hist_grid) split_hist(tb, hist_grid);
    if (static_cast<size_t>(blockIdx.x) * kNT < n) scan_block_sum(cc, tb.scan_tmp);   // block-uniform
}

// Largest box extent a walk group of system s may have: efac x the cell side
// at the first depth whose non-empty cells number at least n_s / occ (with
// occ = 32, cells there hold ~32 bodies on average).  A group much wider than
// its neighbours' spacing would force the walk to open everything its box
// overlaps.  Clears dcount for the next step.  Run by block 0 of k_slots,
// the launch after k_split_hist.
__device__ inline void sys_extents(const TreeBuffers& tb, const GroupParams& gp)
{
    for (uint32_t q = threadIdx.x; q < tb.n_sys; q += kNT) {
        SysScalars* sy = tb.sys + q;
        const size_t ns = sy->body_hi - sy->body_lo;
        uint32_t dc[kMaxDepth + 1];   // every depth's count in one round of loads
#pragma unroll
        for (int e = 0; e <= kMaxDepth; ++e) dc[e] = sy->dcount[e];
        uint32_t cells = 1;
        int d = 0;
#pragma unroll
        for (int e = 0; e < kMaxDepth; ++e) {
            if (d == e && static_cast<size_t>(cells) * gp.occ < ns) {
                cells += dc[e];
                d = e + 1;
            }
        }
        sy->emax = gp.efac * sqrt(sy->side2[d]);
#pragma unroll
        for (int e = 0; e <= kMaxDepth; ++e) sy->dcount[e] = 0;
    }
}

__device__ inline double box_extent(const double* bx)
{
    const double e = fmax(bx[3] - bx[0], fmax(bx[4] - bx[1], bx[5] - bx[2]));
    return e > 0.0 ? e : 0.0;   // an empty box (no light bodies) has extent 0
}

// group starts (flags at the first body of every group).  A unit is "good"
// when it holds <= gmax bodies and its light bodies' box is within its
// system's extent limit (a leaf always qualifies); goodness passes to
// children.  Groups are the maximal good units, and runs of good siblings are
// packed while the count fits gmax and their joint box stays within the
// limit.  Everything here depends on the system's bodies alone, so every
// schedule, and every other system of an ensemble, sees the same groups.
// Body i starts a group: its flag, counted in its 256-body tile.  Each body
// is marked by one node at most (the root, the co-keyed leaf that holds it,
// or the parent of the unit it starts), so the count is the tile's flag sum.
__device__ inline void mark_group(const TreeBuffers& tb, uint32_t i)
{
    tb.gflag[i] = 1;
    atomicAdd(tb.gtile + (i >> 8), 1u);
}

__global__ __launch_bounds__(kNT) void k_group_marks(size_t n, TreeBuffers tb, MixedBuffers mb, uint32_t gmax)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    const uint32_t M = tb.sc->n_leaves, B = tb.sc->n_branch;
    if (t >= static_cast<size_t>(M) + B) return;
    const uint32_t u = static_cast<uint32_t>(t);
    // The loads come in dependent rounds, each issued together (the node's
    // leaf range, then its bodies; then, above the groups, every child's
    // range, bodies and box) so that a node costs a few memory trips and not
    // one per child.
    const bool leaf = u < M;
    const uint32_t par = tb.parent[u];
    uint32_t lo = u, hi = u, depth = kMaxDepth;
    if (!leaf) {
        lo = tb.blo[u - M];
        hi = tb.bhi[u - M];
        depth = tb.bdepth[u - M];
    }
    double ub[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) ub[a] = leaf ? 0.0 : tb.lbox[6 * static_cast<size_t>(u) + a];
    const uint32_t f = tb.leaf_first[lo];
    const uint32_t cnt = tb.leaf_first[hi + 1] - f;
    const double emax = tb.sys[tb.n_sys == 1 ? 0u : tb.bsys[f]].emax;
    auto good_box = [&](bool is_leaf, uint32_t cv, const double* bx) {
        return cv <= gmax && (is_leaf || box_extent(bx) <= emax);
    };
    const bool ugood = good_box(leaf, cnt, ub);
    if (par == kNone && ugood) {
        mark_group(tb, f);
        mb.gdepth[f] = static_cast<uint8_t>(depth);
        return;
    }
    if (leaf) {
        if (cnt > gmax) {   // co-keyed bodies beyond one group
            for (uint32_t k = 0; k < cnt; k += gmax) {
                mark_group(tb, f + k);
                mb.gdepth[f + k] = kMaxDepth;
            }
        }
        return;
    }
    if (ugood) return;   // inside a group formed above
    const int4* c4 = reinterpret_cast<const int4*>(tb.child + 8 * static_cast<size_t>(u - M));
    const int4 ca = c4[0], cb = c4[1];
    const int32_t c[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
    // an empty octant reads the node's first leaf and is skipped below
    uint32_t clo[8], chi[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t cv = c[k] < 0 ? lo : static_cast<uint32_t>(c[k]);
        clo[k] = cv < M ? cv : tb.blo[cv - M];
        chi[k] = cv < M ? cv : tb.bhi[cv - M];
    }
    uint32_t cf[8], cc[8];
    double cbx[8][6];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t cv = c[k] < 0 ? lo : static_cast<uint32_t>(c[k]);
        cf[k] = tb.leaf_first[clo[k]];
        cc[k] = tb.leaf_first[chi[k] + 1];
#pragma unroll
        for (int a = 0; a < 6; ++a) cbx[k][a] = tb.lbox[6 * static_cast<size_t>(cv) + a];
    }
    uint32_t cur = 0;
    bool open = false;
    double rl[3] = {0, 0, 0}, ru[3] = {0, 0, 0};   // joint light box of the open run
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (c[k] < 0) continue;
        const uint32_t cv = static_cast<uint32_t>(c[k]);
        const uint32_t ccount = cc[k] - cf[k];
        const double* bx = cbx[k];
        if (!good_box(cv < M, ccount, bx)) {
            open = false;
            continue;
        }
        const bool empty = !(bx[0] <= bx[3]);
        bool fits = open && cur + ccount <= gmax;
        if (fits && !empty) {
            double e = 0.0;
            for (int a = 0; a < 3; ++a) e = fmax(e, fmax(ru[a], bx[3 + a]) - fmin(rl[a], bx[a]));
            fits = e <= emax;
        }
        if (!fits) {
            mark_group(tb, cf[k]);
            mb.gdepth[cf[k]] = static_cast<uint8_t>(depth + 1);
            cur = 0;
            open = true;
            for (int a = 0; a < 3; ++a) {
                rl[a] = INFINITY;
                ru[a] = -INFINITY;
            }
        }
        cur += ccount;
        if (!empty)
            for (int a = 0; a < 3; ++a) {
                rl[a] = fmin(rl[a], bx[a]);
                ru[a] = fmax(ru[a], bx[3 + a]);
            }
    }
}

// A group is shared by a block's wavefronts, and walked first, when its work in
// the previous walk exceeds this: kShare x (groups per wave) x (an even share of
// the walk per wave), see kShareNum; with many groups per wave an eighth of an
// even share and four times the mean, which only the groups of far-apart heavy
// bodies exceed.  (One that starts late ends late: the 64-system ensemble's walk
// 5.6 -> 4.25 ms with two such groups.)
__device__ inline uint64_t share_limit(const StepScalars* sc, uint32_t walk_waves)
{
    const uint64_t even = sc->work_prev / walk_waves;
    const uint64_t many = sc->work_prev * sc->groups_prev * kShareNum / (static_cast<uint64_t>(walk_waves) * walk_waves * kShareDen);
    const uint64_t mean = sc->work_prev / max(sc->groups_prev, 1u);
    return min(many, max(even / 8u, 4u * mean));
}

__device__ inline void group_first(size_t i, size_t n, uint32_t gid, const Bodies& b, const TreeBuffers& tb,
                                   const MixedBuffers& mb)
{
    const uint32_t f = tb.gflag[i];
    if (f) {
        mb.gfirst[gid] = static_cast<uint32_t>(i);
        bool big = tb.sc->work_prev != 0u && b.pcost[i] > share_limit(tb.sc, mb.walk_waves);
        if (big) {
            const uint32_t k = atomicAdd(&tb.sc->n_big, 1u);
            // (at most waves^2 / (kShare x groups) or 8 x waves groups of the previous
            // walk exceed the limit; smaller groups since, each with the work of the
            // group its bodies were in, can be more: the rest are not shared)
            big = k < kMaxShared;
            if (big) mb.chunk[k] = gid;
        }
        mb.gbig[gid] = big ? 1u : 0u;
    }
    if (i + 1 == n) {   // the group count G and the end sentinel gfirst[G] = n
        mb.gfirst[gid + f] = static_cast<uint32_t>(n);
        tb.sc->n_groups = gid + f;
    }
}

// slots: the root of system s at s; children of branching node b at
// n_sys + base[b] + rank, base = the exclusive scan of the child counts.
// Block 0 also sets the systems' extent limits.
__global__ __launch_bounds__(kNT) void k_slots(size_t n, TreeBuffers tb, MixedBuffers mb, GroupParams gp)
{
    const size_t bi = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (blockIdx.x == 0) sys_extents(tb, gp);
    const uint32_t base = scan_block_excl(bi < n ? child_count(tb, bi) : 0u, tb.scan_tmp, n);
    if (bi < n) mb.base[bi] = base;
    if (bi < tb.n_sys) mb.slot[tb.sys[bi].root] = static_cast<uint32_t>(bi);
    if (bi >= tb.sc->n_branch) return;
    const int32_t* ch = tb.child + 8 * bi;
    uint32_t k = 0;
    const uint32_t b0 = tb.n_sys + base;
#pragma unroll
    for (int o = 0; o < 8; ++o)
        if (ch[o] >= 0) mb.slot[ch[o]] = b0 + k++;
}

// thread t: the first body of group t (t < n) and node record t (t < M + B)
__global__ __launch_bounds__(kNT) void k_mixed_nodes(size_t n, Bodies b, TreeBuffers tb, MixedBuffers mb, double G)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (static_cast<size_t>(blockIdx.x) * kNT < n) {   // block-uniform: the blocks over the bodies
        const uint32_t gid = scan_block_excl(t < n ? tb.gflag[t] : 0u, tb.gtile, n);
        if (t < n) group_first(t, n, gid, b, tb, mb);
    }
    const uint32_t M = tb.sc->n_leaves, B = tb.sc->n_branch;
    if (t >= static_cast<size_t>(M) + B) return;
    // every load that needs no loaded value first, in one round: the light
    // moments, box and slot, and the leaf's body range or the node's children
    const double* q = tb.lraw + 4 * t;
    const double m = q[0], q1 = q[1], q2 = q[2], q3 = q[3], sec = tb.lsec[t];
    double bx[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) bx[a] = tb.lbox[6 * t + a];
    const uint32_t slot = mb.slot[t];
    const bool leaf = t < M;
    uint32_t f0 = 0, f1 = 0, base = 0;
    int4 ca = make_int4(-1, -1, -1, -1), cb = ca;
    if (leaf) {
        f0 = tb.leaf_first[t];
        f1 = tb.leaf_first[t + 1];
    } else {
        const int4* c4 = reinterpret_cast<const int4*>(tb.child + 8 * (t - M));
        ca = c4[0];
        cb = c4[1];
        base = mb.base[t - M];
    }
    MNode nd;
    if (m != 0.0) {
        nd.x = q1 / m;
        nd.y = q2 / m;
        nd.z = q3 / m;
    } else {
        nd.x = nd.y = nd.z = 0.0;
    }
    nd.gm = static_cast<float>(G * m);
    // Q = sum m |x - com|^2 = sum m |x|^2 - |sum m x|^2 / m; the cancellation
    // costs (|x| / extent)^2 ulps, harmless for an opening test
    const double quad = m != 0.0 ? sec - (q1 * q1 + q2 * q2 + q3 * q3) / m : 0.0;
    nd.gq = static_cast<float>(G * (quad > 0.0 ? quad : 0.0));
    // opening size: the farthest corner of the light bodies' box seen from the
    // centre of mass (0 for an empty node)
    double s2 = 0.0;
    if (m != 0.0) {
        const double c3[3] = {nd.x, nd.y, nd.z};
        for (int a = 0; a < 3; ++a) {
            const double e = fmax(c3[a] - bx[a], bx[3 + a] - c3[a]);
            s2 += e * e;
        }
    }
    nd.size2 = s2;
    if (leaf) {
        nd.push = stack_range(f0, f1 - f0, true);
        nd.info = (f1 - f0) | kMLeaf;
        if (f1 - f0 > 1u) nd.size2 = INFINITY;
        else {
            // the body itself (its light mass is its mass, or 0 if heavy):
            // the walk appends it from the node alone, with the very offsets
            // a body entry gives, which the self-term test relies on
            nd.x = b.px[f0];
            nd.y = b.py[f0];
            nd.z = b.pz[f0];
        }
    } else {
        const int32_t c[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
        uint32_t k = 0;
#pragma unroll
        for (int o = 0; o < 8; ++o) k += c[o] >= 0 ? 1u : 0u;
        nd.push = stack_range(tb.n_sys + base, k, false);
        nd.info = k;
    }
    mb.node[slot] = nd;
}

// ------------------------------------------------------------- walk
__device__ inline uint32_t uni(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

// Cross-lane moves within a row of 16 lanes by DPP (no LDS round trip);
// kCtrl: 0x120 + k rotates the row right by k, 0x110 + k shifts it right
template <int kCtrl>
__device__ inline double dpp_f64(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), kCtrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), kCtrl, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

__device__ inline double min2(double v, double t) { return (t < v) ? t : v; }
__device__ inline double max2(double v, double t) { return (v < t) ? t : v; }

__device__ inline double wave_min(double v)
{
    v = min2(v, dpp_f64<0x128>(v));
    v = min2(v, dpp_f64<0x124>(v));
    v = min2(v, dpp_f64<0x122>(v));
    v = min2(v, dpp_f64<0x121>(v));
    v = min2(v, __shfl_xor(v, 16, 64));
    return min2(v, __shfl_xor(v, 32, 64));
}
__device__ inline double wave_max(double v)
{
    v = max2(v, dpp_f64<0x128>(v));
    v = max2(v, dpp_f64<0x124>(v));
    v = max2(v, dpp_f64<0x122>(v));
    v = max2(v, dpp_f64<0x121>(v));
    v = max2(v, __shfl_xor(v, 16, 64));
    return max2(v, __shfl_xor(v, 32, 64));
}

// lane k's value (k wave-uniform)
__device__ inline uint32_t lane_u32(uint32_t v, uint32_t k)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(k)));
}
__device__ inline double lane_f64(double v, uint32_t k)
{
    const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
    const uint64_t lo = lane_u32(static_cast<uint32_t>(u), k), hi = lane_u32(static_cast<uint32_t>(u >> 32), k);
    return __longlong_as_double(static_cast<long long>((hi << 32) | lo));
}

// number of set lanes of mask below this lane
__device__ inline uint32_t rank_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

__device__ inline uint32_t wave_incl_scan(uint32_t v)
{
    // rows of 16 by row shifts, then row 0 into row 1 and 2 into 3, then the
    // lower half into the upper (row_bcast); absent lanes add 0
    int x = static_cast<int>(v);
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return static_cast<uint32_t>(x);
}

struct Acc3 {
    float sx = 0.f, sy = 0.f, sz = 0.f;   // Kahan sums
    float cx = 0.f, cy = 0.f, cz = 0.f;   // compensations
    __device__ static void kadd(float& s, float& c, float v)
    {
        const float y = v - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    __device__ void add(float bx, float by, float bz)
    {
        kadd(sx, cx, bx);
        kadd(sy, cy, by);
        kadd(sz, cz, bz);
    }
};

// The r^2 every list interaction starts from: the softening, but at least
// 1e-24 x max(1, (G M)^(2/3)) for the light mass G M of the group's system.
// The self entry (the lane's own body: dx = dy = dz = 0 exactly) then has
// rsq <= 1e12 / max(1, (G M)^(1/3)) and G m rsq^3 <= 1e36, so it adds
// 0 * finite = +0 with no clamp in the loop.  Another pair's r^2 moves by at
// most the floor, below half an ulp once r^2 exceeds 2^25 x the floor
// (a distance of 6e-9 in a system with G M <= 1).
__device__ inline float list_r2_floor(float gm, float soft2)
{
    const float e = gm > 1.f ? exp2f((2.f / 3.f) * log2f(gm)) : 1.f;
    return fmaxf(soft2, 1e-24f * e);
}

// r2_0 is list_r2_floor's value: with it every r2 is positive and every
// rsq finite
__device__ inline void interact(const float4 q, float ox, float oy, float oz, float r2_0, float& bx, float& by,
                                float& bz)
{
    const float dx = q.x - ox;
    const float dy = q.y - oy;
    const float dz = q.z - oz;
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, r2_0)));
    const float inv = __builtin_amdgcn_rsqf(r2);
    const float s = q.w * (inv * inv * inv);
    bx = fmaf(s, dx, bx);
    by = fmaf(s, dy, by);
    bz = fmaf(s, dz, bz);
}

// ------------------------------------------------- evaluating the list
// A group of cnt bodies has S partial sums per body (list_shares), and the
// list of a flush is cut into S shares of len consecutive entries
// (share_len).  Virtual lane t = s cnt + b takes share s for body b, so 128
// or 256 virtual lanes hold a group whatever its size; a wavefront (NW = 1)
// runs them as up to four passes over the list, a block of NW wavefronts as
// 4 / NW passes each.  Every virtual lane's sum -- FP32 FMA over blocks of 32
// entries, Kahan-compensated across blocks and flushes -- depends on the
// group alone, so every NW gives the same bits.  Against idle lanes taking
// over stretches of other lanes' bodies (which this replaced) the wave steps
// are 2% fewer (1.085 against 1.106 x the ideal on a 300k belt), with no
// hand-over.
__device__ inline uint32_t list_shares(uint32_t cnt)
{
    const uint32_t s = (cnt <= 16u ? 128u : 256u) / cnt;
    return s > 32u ? 32u : s;
}

// Entries per share: at least ceil(ln / S), and a length whose multiples fall
// into different LDS banks for the shares that meet in one wavefront (16
// entries of 16 bytes span all banks): odd for small groups, whose
// wavefronts mix many shares, else no multiple of 8.  invS = ceil(65536 / S):
// the quotient is exact for ln < 330 and S <= 32.  S len <= kListCap + kListPad.
__device__ inline uint32_t share_len(uint32_t ln, uint32_t S, uint32_t invS, uint32_t cnt)
{
    const uint32_t len = ((ln + S - 1u) * invS) >> 16;
    if (cnt <= 16u) return len | 1u;
    return (cnt < 64u && (len & 7u) == 0u) ? len + 1u : len;
}

template <int N>
__device__ inline void interact_n(const float4* __restrict__ p, float ox, float oy, float oz, float r2_0, float& bx,
                                  float& by, float& bz)
{
    float4 q[N];
#pragma unroll
    for (int k = 0; k < N; ++k) q[k] = p[k];
#pragma unroll
    for (int k = 0; k < N; ++k) interact(q[k], ox, oy, oz, r2_0, bx, by, bz);
}

// p[0..len) (len wave-uniform) for one body: blocks of 32 entries, eight
// loaded at a time, each block's FP32 sum added into a
__device__ inline void share_sum(const float4* __restrict__ p, uint32_t len, float ox, float oy, float oz, float r2_0,
                                 Acc3& a)
{
    uint32_t j = 0;
    while (j < len) {
        const uint32_t end = min(len, j + 32u);
        float bx = 0.f, by = 0.f, bz = 0.f;
        for (; j + 8u <= end; j += 8u) interact_n<8>(p + j, ox, oy, oz, r2_0, bx, by, bz);
        if (end - j >= 4u) {
            interact_n<4>(p + j, ox, oy, oz, r2_0, bx, by, bz);
            j += 4u;
        }
        if (end - j >= 2u) {
            interact_n<2>(p + j, ox, oy, oz, r2_0, bx, by, bz);
            j += 2u;
        }
        if (end - j >= 1u) {
            interact_n<1>(p + j, ox, oy, oz, r2_0, bx, by, bz);
            j += 1u;
        }
        a.add(bx, by, bz);
    }
}

// The schedules' cost of a flushed list of ln entries, in wave steps of one
// wavefront with 4, 2 or 1 lanes per body; for 33..63 bodies only the entries
// beyond the stretches that idle lanes can take over count.  (Chosen by
// measurement on the 300k learned step: counting every step ordered the
// groups 1% worse, the whole list 1.5% worse.)
constexpr uint32_t kMinShare = 32;   // shortest stretch, in entries, that counts as taken over
__device__ inline uint32_t list_cost(uint32_t ln, uint32_t cnt)
{
    if (cnt <= 16u) return (ln + 3u) >> 2;
    if (cnt <= 32u) return (ln + 1u) >> 1;
    const uint32_t E = 64u - cnt;
    if (E == 0u) return ln;
    const uint32_t q = (cnt + E - 1u) / E;
    const uint32_t R = (ln / (q + 1u)) & ~7u;
    return R < kMinShare ? ln : ln - q * R;
}

// A round's ranges, one per lane in the order of the pop: range r holds the
// slots [excl, excl + count) of the round, and its slot s stands for the node
// (or body) info + s.
struct Ranges {
    uint32_t info, excl, count, total;   // total: the round's slots (wave-uniform)
};
constexpr int kRoundSlots = 512;   // 64 ranges of at most 8

// A lone wavefront writes out the entries of a whole round at once ...
__device__ inline void write_slots(const Ranges& r, uint32_t* slots)
{
    const uint32_t e = r.info + r.excl;
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k)
        if (k < r.count) slots[r.excl + k] = e + k;
    __builtin_amdgcn_wave_barrier();
}

// ... wavefronts that share a round find each of their own 64: the entry of
// slot sb + lane belongs to the last range that starts at or before it, found
// by marking the starts that fall into the 64 slots (mark: 64 words of the
// wavefront's own) and a running maximum of their lanes.
__device__ inline uint32_t slot_entry(const Ranges& r, uint32_t sb, uint32_t* mark)
{
    const uint32_t lane = __lane_id();
    const uint32_t at = r.excl - sb;
    const uint32_t before = static_cast<uint32_t>(__popcll(__ballot(r.count != 0u && r.excl < sb)));
    mark[lane] = 0u;
    __builtin_amdgcn_wave_barrier();
    if (r.count != 0u && at < 64u) mark[at] = lane + 1u;
    __builtin_amdgcn_wave_barrier();
    int x = static_cast<int>(mark[lane]);
    __builtin_amdgcn_wave_barrier();
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));
    x = max(x, static_cast<int>(before));
    const uint32_t s = sb + lane;
    const uint32_t e = static_cast<uint32_t>(__shfl(static_cast<int>(r.info), x - 1, 64)) + s;
    return s < r.total ? e : 0u;
}

// Entry of slot sb + lane (0 past the round's end) and its node, a zero node
// (no mass: never used) for a body entry and past the end.
template <int NW>
__device__ inline uint32_t fetch_slot(const Ranges& r, uint32_t sb, uint32_t* slots, const MNode* __restrict__ nodes,
                                      MNode& nd)
{
    const uint32_t s = sb + __lane_id();
    uint32_t ent = 0u;
    if (NW == 1) {
        if (s < r.total) ent = slots[s];
    } else {
        ent = slot_entry(r, sb, slots);
    }
    nd = MNode{};
    if (s < r.total && !(ent & 0x80000000u)) nd = nodes[ent];
    return ent;
}

// Waits for the block's other wavefronts; a lone wavefront needs no
// barrier (its LDS accesses stay in order), only that the compiler keeps them
// in place.
template <int NW>
__device__ inline void group_sync()
{
    if (NW == 1) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
}

// Key order: entry t of part x is group (t / R * P + x) * R + t % R, increasing
// in t, so the first t past the end closes x.  The part's blocks hold its first
// part_blocks entries; the queue hands out the rest.
__device__ inline uint32_t part_group(uint32_t x, uint32_t t)
{
    const uint64_t q = (static_cast<uint64_t>(t / kWalkRun) * kWalkParts + x) * kWalkRun + t % kWalkRun;
    return q < kNone ? static_cast<uint32_t>(q) : kNone;
}
__device__ inline uint32_t part_blocks(uint32_t x, uint32_t nblk)
{
    return nblk > x ? (nblk - x + kWalkParts - 1) / kWalkParts : 0u;
}

// Accelerations of the heavy bodies: an FP64 direct sum over every other
// body (compensated per thread, partials combined in thread order).
// The heavy bodies are few and their net accelerations are small next to the
// forces that cancel in them, so no tree truncation is taken for them.

// 1 / sqrt(x) for x > 0: the hardware estimate refined by two Newton steps
// y <- y (3/2 - x/2 y^2), each of which squares the relative error, instead
// of a square root followed by a division (two long dependent sequences)
__device__ inline double rsqrt_f64(double x)
{
    const double hx = 0.5 * x;
    double y = __builtin_amdgcn_rsq(x);
    y = y * (1.5 - hx * y * y);
    y = y * (1.5 - hx * y * y);
    return y;
}

// A partial sum (system s, heavy rank k, chunk c) is heavy body k of system s
// summed over the c-th run of 1024 bodies of s by one wavefront -- each lane
// a compensated sum over its stride, lane partials added in lane order -- and
// k_heavy_final adds the chunk partials in chunk order.  A system's heavy
// accelerations therefore depend on that system alone, not on the launch
// shape or on the other systems of an ensemble.
// A work item is kHeavyTogether ranks of a chunk: a body is loaded once for
// all of them (one rank at a time read every body 16 times a step, 2.1 GB at
// 4M bodies), and items in a row are the ranks of one chunk.  (In a launch of
// their own: 4M bodies 0.307 -> 0.141 ms, 1M 0.068 -> 0.040; the FP64 work of
// the pairs is 0.09 ms at 4M.)
constexpr uint32_t kHeavyTogether = 4;
static_assert(kMaxHeavy % kHeavyTogether == 0, "whole items");
constexpr uint32_t kHeavyRow = 65;   // lane partials of a sum, padded for the banks
struct HeavyArgs {
    const double *px, *py, *pz, *m;
    const SysScalars* sys;
    uint32_t n_sys;
    double* hpart;
    double soft2, G;
};

__device__ inline void heavy_item(const HeavyArgs& ha, uint32_t item, int lane, double (*part)[kHeavyRow])
{
    uint32_t lo = 0, hi = ha.n_sys;   // the last system whose first item is <= item
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (ha.sys[mid].heavy_item / kHeavyTogether <= item) lo = mid;
        else hi = mid;
    }
    const SysScalars* sy = ha.sys + lo;
    const uint32_t r = item - sy->heavy_item / kHeavyTogether;
    constexpr uint32_t kSets = kMaxHeavy / kHeavyTogether;
    const uint32_t k0 = r % kSets * kHeavyTogether, c = r / kSets, nh = sy->n_heavy;
    if (k0 >= nh) return;
    uint32_t h[kHeavyTogether];
    double x[kHeavyTogether], y[kHeavyTogether], z[kHeavyTogether];
    ExactSum a[kHeavyTogether][3];
#pragma unroll
    for (uint32_t q = 0; q < kHeavyTogether; ++q) {
        h[q] = sy->heavy_slot[min(k0 + q, nh - 1)];
        x[q] = ha.px[h[q]];
        y[q] = ha.py[h[q]];
        z[q] = ha.pz[h[q]];
    }
    const size_t j0 = sy->body_lo + static_cast<size_t>(c) * kHeavyChunk;
    const size_t j1 = min(j0 + kHeavyChunk, static_cast<size_t>(sy->body_hi));
    // the heavy body itself and co-located bodies add an exact zero (a no-op
    // for the sums) instead of being skipped, so the loop unrolls and the
    // square roots of consecutive bodies overlap
#pragma unroll 2
    for (size_t j = j0 + lane; j < j1; j += 64) {
        const double bx = ha.px[j], by = ha.py[j], bz = ha.pz[j], gm = ha.G * ha.m[j];
#pragma unroll
        for (uint32_t q = 0; q < kHeavyTogether; ++q) {
            const double dx = bx - x[q], dy = by - y[q], dz = bz - z[q];
            const double r2 = dx * dx + dy * dy + dz * dz + ha.soft2;
            const double invR = rsqrt_f64(r2);
            const double s = (j != h[q] && r2 > 0.0) ? gm * (invR * invR * invR) : 0.0;
            a[q][0].add(s * dx);
            a[q][1].add(s * dy);
            a[q][2].add(s * dz);
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < kHeavyTogether; ++q)
#pragma unroll
        for (int d = 0; d < 3; ++d) part[3 * q + d][lane] = a[q][d].value();
    __builtin_amdgcn_wave_barrier();
    const uint32_t k = k0 + static_cast<uint32_t>(lane) / 3u;
    if (lane < 3 * static_cast<int>(kHeavyTogether) && k < nh) {
        ExactSum t;
        for (int q = 0; q < 64; ++q) t.add(part[lane][q]);
        ha.hpart[3 * (sy->heavy_item + static_cast<size_t>(k) * sy->heavy_chunks + c) + lane % 3] = t.value();
    }
    __builtin_amdgcn_wave_barrier();
}

// The walk of a group, by one wavefront (NW = 1) or by the four of a block
// (NW = 4): each round's nodes 64 per wavefront, the list's virtual lanes 64
// per wavefront.  The order of the nodes, the list and its flushes, and every
// sum are the same for both, so the results are the same bits.
//
// The arguments (some 70 pointers and scalars) are read from the kernel's
// argument segment where a stage needs them: held in scalar registers across
// the whole loop they were spilled to vector registers (100 spills).
struct WalkArgs {
    Bodies b;
    TreeBuffers tb;
    MixedBuffers mb;
    MixedParams p;
};
using WalkArgsP = const __attribute__((address_space(4))) WalkArgs*;

// the arguments, read again after this point (the compiler cannot tell that
// the address is the same, so it does not keep earlier loads alive)
__device__ inline WalkArgsP args_here(WalkArgsP a)
{
    asm volatile("" : "+s"(a));
    return a;
}

// Body j as a list entry of a group centred on (cx, cy, cz); false (q left
// alone) for a heavy or massless body.
__device__ inline bool body_entry(WalkArgsP a, uint32_t j, double cx, double cy, double cz, float4& q)
{
    const double m = a->b.m[j];
    if (a->b.hrank[j] >= 0 || m == 0.0) return false;
    q = make_float4(static_cast<float>(a->b.px[j] - cx), static_cast<float>(a->b.py[j] - cy),
                    static_cast<float>(a->b.pz[j] - cz), static_cast<float>(a->p.G * m));
    return true;
}

// LDS of a block: four wavefronts' own, or one shared group's, over it.
// The list (with its padding), then the words of write_slots or 64 per
// wavefront for slot_entry, then the stack; the sums that are exchanged (256
// doubles, 768 between wavefronts) lie over the first two.
constexpr int kListBytes = (kListCap + kListPad) * 16;
constexpr int kWaveLds = kListBytes + kRoundSlots * 4 + kStackCap * 4;
static_assert(kListBytes + kRoundSlots * 4 >= 768 * 8, "the exchanged sums fit");
static_assert(kWaveLds >= 3 * kHeavyTogether * kHeavyRow * 8, "a heavy item's lane partials fit");

// Walks group g by NW wavefronts (1: this one alone; 4: the block's, this one
// the w-th) and returns its work.  turn_no: exchanges so far (which of the two
// rows of s_word is next).
template <int NW>
__device__ __forceinline__ uint32_t walk_group(WalkArgsP args, StepScalars* sc, uint32_t g, int w, int lane,
                                           unsigned char* lds, uint32_t (*s_word)[kWaves], uint32_t& turn_no)
{
    constexpr int V = 4 / NW;   // passes over a list: virtual wavefronts w, w + NW, ... of the group's four
    const uint32_t tid = static_cast<uint32_t>(w * 64 + lane);
    float4* list = reinterpret_cast<float4*>(lds);
    uint32_t* slots = reinterpret_cast<uint32_t*>(lds + kListBytes) + w * 64;
    uint32_t* stk = reinterpret_cast<uint32_t*>(lds + kListBytes + kRoundSlots * 4);
    double* part_sum = reinterpret_cast<double*>(lds);
    const uint64_t t_start = wall_clock64();
    const WalkArgsP ag = args_here(args);
    const uint32_t b0 = uni(ag->mb.gfirst[g]);
    const uint32_t cnt = uni(ag->mb.gfirst[g + 1]) - b0;
    // lane = body for the box, the heavy bodies and the results
    const bool valid = static_cast<uint32_t>(lane) < cnt;
    const uint32_t i = b0 + (valid ? static_cast<uint32_t>(lane) : 0u);
    const double x = ag->b.px[i], y = ag->b.py[i], z = ag->b.pz[i];
    // virtual lanes: share and body of pass v (share >> 8 | body; a lane
    // past the last share repeats share 0 and its sum is never read)
    const uint32_t S = list_shares(cnt), invS = (65535u + S) / S;
    uint32_t vl[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const uint32_t t = static_cast<uint32_t>((v * NW + w) * 64 + lane);
        const uint32_t sh = t / cnt;
        vl[v] = (t - sh * cnt) | ((sh < S ? sh : 0u) << 8);
    }
    const double lox = wave_min(x), loy = wave_min(y), loz = wave_min(z);
    const double hix = wave_max(x), hiy = wave_max(y), hiz = wave_max(z);
    const double cx = 0.5 * (lox + hix), cy = 0.5 * (loy + hiy), cz = 0.5 * (loz + hiz);
    const double hx = 0.5 * (hix - lox), hy = 0.5 * (hiy - loy), hz = 0.5 * (hiz - loz);
    const float ox = static_cast<float>(x - cx);
    const float oy = static_cast<float>(y - cy);
    const float oz = static_cast<float>(z - cz);
    Acc3 acc[V];
    uint32_t ln = 0, sp = 1, n_inter = 0, n_visit = 0, n_steps = 0;
    bool overflow = false;
    const uint32_t gsys = ag->tb.n_sys == 1 ? 0u : uni(ag->tb.bsys[b0]);
    const MNode* __restrict__ nodes = ag->mb.node;
    const float r2_0 = list_r2_floor(nodes[gsys].gm, static_cast<float>(ag->p.soft2));   // the system's root
    // heavy bodies of the system: FP64 direct sum, the ranks k = q mod 4 in
    // rank order into partial q (one or more of the four per wavefront),
    // the partials added in order
    double hax = 0.0, hay = 0.0, haz = 0.0;
    {
        const SysScalars* sy = ag->tb.sys + gsys;
        const uint32_t nh = sy->n_heavy;
        const double soft2 = ag->p.soft2, grav = ag->p.G;
        // lane k loads heavy body k (one load latency for all of them); the
        // loop reads them back as wave constants
        uint32_t hj = kNone;
        double hpx = 0.0, hpy = 0.0, hpz = 0.0, hpm = 0.0;
        if (static_cast<uint32_t>(lane) < nh) {
            hj = sy->heavy_slot[lane];
            hpx = ag->b.px[hj];
            hpy = ag->b.py[hj];
            hpz = ag->b.pz[hj];
            hpm = ag->b.m[hj];
        }
#pragma unroll 1
        for (int v = 0; v < V; ++v) {
            double sx = 0.0, sy_ = 0.0, sz = 0.0;
            for (uint32_t k = static_cast<uint32_t>(v * NW + w); k < nh; k += 4u) {
                const uint32_t j = lane_u32(hj, k);
                const double dx = lane_f64(hpx, k) - x, dy = lane_f64(hpy, k) - y, dz = lane_f64(hpz, k) - z;
                const double r2 = dx * dx + dy * dy + dz * dz + soft2;
                const bool pair = j != i && r2 > 0.0;
                const double invR = __all(inv_sqrt_takes(r2) | !pair) ? inv_sqrt_in_range(pair ? r2 : 1.0)
                                                                      : 1.0 / sqrt(pair ? r2 : 1.0);
                const double s = grav * lane_f64(hpm, k) * (invR * invR * invR);
                if (pair) {
                    sx += s * dx;
                    sy_ += s * dy;
                    sz += s * dz;
                }
            }
            if (NW == 1) {
                hax += sx;
                hay += sy_;
                haz += sz;
            } else {
                double* q = part_sum + (v * NW + w) * 192 + lane;
                q[0] = sx;
                q[64] = sy_;
                q[128] = sz;
            }
        }
    }
    if (NW > 1) {
        __syncthreads();
        for (int q = 0; q < 4; ++q) {
            hax += part_sum[q * 192 + lane];
            hay += part_sum[q * 192 + 64 + lane];
            haz += part_sum[q * 192 + 128 + lane];
        }
    }
    // relative opening test: a node is also opened while its quadrupole
    // scale G Q / D^4 exceeds alpha x the smallest heavy-body acceleration
    // of the group (the acceleration every body of these systems is made of)
    const double ah = valid ? sqrt(hax * hax + hay * hay + haz * haz) : INFINITY;
    const double aref = wave_min(ah);
    const double alpha = ag->p.alpha, theta2 = ag->p.theta2;
    const double qlim = (alpha > 0.0 && aref > 0.0 && aref < INFINITY) ? alpha * aref : INFINITY;
    // up to theta^2 = kSafe2 (and without a limit) the extent test implies the rest
    const bool relative = theta2 > kSafe2 && __any(qlim < INFINITY);
    bool deep = false;      // the stack was over kNarrowRoom
    bool recount = false;   // the second pass of a training walk
    if (tid == 0) stk[0] = stack_range(gsys, 1, false);   // the root of the group's system
    group_sync<NW>();   // (also: every wavefront has read the exchanged sums)
    for (bool last = false; !last;) {
        // pop up to 64 ranges, one per lane, while the stack cannot
        // overflow; when it is empty one more turn flushes the rest of the list
        last = sp == 0u || overflow;
        Ranges r{0u, 0u, 0u, 0u};
        if (!last) {
            deep |= sp > kNarrowRoom;
            const uint32_t P = pop_count(sp, recount);
            const bool has = static_cast<uint32_t>(lane) < P;
            const uint32_t e = has ? stk[sp - 1 - lane] : 0u;
            sp -= P;
            r.count = has ? ((e >> 27) & 7u) + 1u : 0u;
            const uint32_t incl = wave_incl_scan(r.count);
            r.total = lane_u32(incl, 63);
            r.excl = incl - r.count;
            r.info = (e & 0x87ffffffu) - r.excl;
            n_visit += r.total;
            if (NW == 1) write_slots(r, slots);
        }
        uint32_t ent = 0u;
        MNode nd{};
        if (static_cast<uint32_t>(w) * 64u < r.total) ent = fetch_slot<NW>(r, static_cast<uint32_t>(w) * 64u, slots, nodes, nd);
        uint32_t base = 0;
        do {
            // the opening test; a leaf of one body is always accepted, one
            // of several never (its bodies are), and lanes without a node
            // have no mass
            const double rx = nd.x - cx, ry = nd.y - cy, rz = nd.z - cz;
            const double ex = fmax(fabs(rx) - hx, 0.0);
            const double ey = fmax(fabs(ry) - hy, 0.0);
            const double ez = fmax(fabs(rz) - hz, 0.0);
            const double d2 = ex * ex + ey * ey + ez * ez;
            bool pass = nd.size2 < theta2 * d2;
            if (relative) pass &= nd.size2 <= kSafe2 * d2 || static_cast<double>(nd.gq) <= qlim * (d2 * d2);
            const bool live = nd.gm != 0.f;
            const uint32_t push = nd.push, info = nd.info;
            bool app = live && (pass || info == (kMLeaf | 1u));
            const bool open = live && !app;
            const bool open_big = open && info > (kMLeaf | 8u);
            float4 q = make_float4(static_cast<float>(rx), static_cast<float>(ry), static_cast<float>(rz), nd.gm);
            if (static_cast<int32_t>(ent) < 0) app = body_entry(args_here(args), ent & 0x7fffffffu, cx, cy, cz, q);
            // the next chunk's nodes are on their way while this chunk is
            // listed (without the prefetch: +4% on the 300k walk)
            const uint32_t sb_n = base + static_cast<uint32_t>((NW + w) * 64);
            ent = 0u;
            nd.gm = 0.f;
            if (sb_n < r.total) ent = fetch_slot<NW>(r, sb_n, slots, nodes, nd);
            // list entries and stack pushes of this chunk (one per lane at
            // most), and leaves of more than 8 co-keyed bodies (see below)
            uint64_t am = __ballot(app);
            const uint64_t pm = __ballot(open && !open_big);
            uint64_t big = __ballot(open_big);
            // counts: entries | pushes << 10 | chunks with such leaves << 20,
            // of all NW chunks and of those before this wavefront's
            const uint32_t word = static_cast<uint32_t>(__popcll(am)) |
                                  static_cast<uint32_t>(__popcll(pm)) << 10 | (big ? 1u << 20 : 0u);
            uint32_t all = word, before = 0;
            uint32_t* const row = s_word[turn_no & 1u];
            if (NW > 1) {
                if (lane == 0) row[w] = word;
                __syncthreads();
                ++turn_no;
                all = 0;
#pragma unroll
                for (int c = 0; c < NW; ++c) {
                    const uint32_t v = row[c];
                    before += c < w ? v : 0u;
                    all += v;
                }
                all = uni(all);
                before = uni(before);
            }
            const uint32_t need = (all >> 10) & 0x3ffu;
            if (sp + need > static_cast<uint32_t>(kStackCap)) {
                if (tid == 0) atomicOr(&sc->error, kErrStack);
                overflow = true;
            } else {
                // one range per opened node or leaf of at most 8 bodies
                if (open && !open_big) stk[sp + ((before >> 10) & 0x3ffu) + rank_below(pm)] = push;
                sp += need;
            }
            if (!last && all < (1u << 20) && ln + (all & 0x3ffu) <= static_cast<uint32_t>(kListCap)) {
                if (app) list[ln + (before & 0x3ffu) + rank_below(am)] = q;
                ln += all & 0x3ffu;
                n_inter += all & 0x3ffu;
            } else {
                // The list is flushed before the chunk that does not fit (and
                // at the end).  A leaf of more than 8 co-keyed bodies
                // (duplicate or nearly coincident positions) puts its bodies
                // on the list directly, 64 at a time, so the stack does not
                // grow with its size: while a round holds such leaves its
                // chunks take turns, wavefront `turn` appending its entries,
                // then its leaves' bodies.
                const bool turns = all >= (1u << 20);
                uint32_t turn = 0, big_k0 = 0;
                for (bool more = true, first = true; more; first = false) {
                    uint32_t words[NW];   // entries of each chunk, | 1 << 20 while its leaves have bodies left
                    const bool mine = !turns || turn == static_cast<uint32_t>(w);
                    am = __ballot(app && mine);
                    if (NW == 1) {
                        words[0] = static_cast<uint32_t>(__popcll(am)) | (big ? 1u << 20 : 0u);
                    } else if (first) {
#pragma unroll
                        for (int c = 0; c < NW; ++c)
                            words[c] = !turns || c == 0 ? uni(row[c]) & 0x1003ffu : 0u;
                    } else {
                        uint32_t* const rw = s_word[turn_no & 1u];
                        if (lane == 0)
                            rw[w] = static_cast<uint32_t>(__popcll(am)) | (mine && big ? 1u << 20 : 0u);
                        __syncthreads();
                        ++turn_no;
#pragma unroll
                        for (int c = 0; c < NW; ++c) words[c] = uni(rw[c]);
                    }
                    for (int c0 = 0;;) {
                        uint32_t l1 = ln, at = 0;
                        int c1 = c0;
#pragma unroll
                        for (int c = 0; c < NW; ++c) {
                            if (c >= c0 && c == c1 && l1 + (words[c] & 0x3ffu) <= static_cast<uint32_t>(kListCap)) {
                                if (c == w) at = l1;
                                l1 += words[c] & 0x3ffu;
                                ++c1;
                            }
                        }
                        if (w >= c0 && w < c1 && ((am >> lane) & 1u)) list[at + rank_below(am)] = q;
                        n_inter += l1 - ln;
                        ln = l1;
                        c0 = c1;
                        if (c0 == NW && !last) break;
                        // flush: padded with entries of no mass to S shares
                        const uint32_t len = share_len(ln, S, invS, cnt);
                        if (tid < 64 && ln + static_cast<uint32_t>(lane) < S * len)
                            list[ln + static_cast<uint32_t>(lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
                        group_sync<NW>();
#pragma unroll
                        for (int v = 0; v < V; ++v) {
                            if (!recount && static_cast<uint32_t>((v * NW + w) * 64) < S * cnt) {
                                const int src = static_cast<int>(vl[v] & 0xffu);
                                share_sum(list + (vl[v] >> 8) * len, len, __shfl(ox, src, 64), __shfl(oy, src, 64),
                                          __shfl(oz, src, 64), r2_0, acc[v]);
                            }
                        }
                        n_steps += list_cost(ln, cnt);
                        group_sync<NW>();
                        ln = 0;
                        if (c0 == NW) break;
                    }
                    more = turns;
                    if (turns) {
                        // the next 64 bodies of this turn's leaves, or the next turn
                        if ((words[turn] >> 20) != 0u) {
                            if (turn == static_cast<uint32_t>(w)) {
                                const uint32_t l = static_cast<uint32_t>(__builtin_ctzll(big));
                                const uint32_t j0 = lane_u32(push, l) & 0x07ffffffu, c = lane_u32(info, l) & ~kMLeaf;
                                const uint32_t j = j0 + big_k0 + static_cast<uint32_t>(lane);
                                app = j < j0 + c && body_entry(args_here(args), j, cx, cy, cz, q);
                                big_k0 += 64u;
                                if (big_k0 >= c) {
                                    big_k0 = 0;
                                    big &= big - 1;
                                }
                            }
                        } else {
                            more = ++turn < static_cast<uint32_t>(NW);
                        }
                    }
                }
            }
            base += NW * 64u;
        } while (base < r.total && !overflow);
        if (last && deep && !recount && !overflow && args_here(args)->p.count_narrow != 0) {
            last = false;
            recount = true;
            sp = 1u;
            n_inter = n_visit = n_steps = 0u;
            if (tid == 0) stk[0] = stack_range(gsys, 1, false);
        }
        group_sync<NW>();   // the next round reads the stack
    }
    // the virtual lanes' sums (a Kahan sum's value is s - c: c holds the
    // negative of the rounding lost), added in FP64 in share order
    double lacc[3];
    if (NW == 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int v = 0; v < V; ++v)
                part_sum[v * 64 + lane] = static_cast<double>(a == 0 ? acc[v].sx : (a == 1 ? acc[v].sy : acc[v].sz)) -
                                          static_cast<double>(a == 0 ? acc[v].cx : (a == 1 ? acc[v].cy : acc[v].cz));
            __builtin_amdgcn_wave_barrier();
            double t = 0.0;
            for (uint32_t k = 0; k < S; ++k) t += part_sum[k * cnt + (valid ? lane : 0)];
            lacc[a] = t;
            __builtin_amdgcn_wave_barrier();
        }
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            double* q = part_sum + (v * NW + w) * 64 + lane;
            q[0] = static_cast<double>(acc[v].sx) - static_cast<double>(acc[v].cx);
            q[256] = static_cast<double>(acc[v].sy) - static_cast<double>(acc[v].cy);
            q[512] = static_cast<double>(acc[v].sz) - static_cast<double>(acc[v].cz);
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            double t = 0.0;
            if (a % NW == w)
                for (uint32_t k = 0; k < S; ++k) t += part_sum[a * 256 + k * cnt + (valid ? lane : 0)];
            lacc[a] = t;
        }
    }
    // heavy bodies take their accelerations from k_heavy_final instead;
    // axis a is written by wavefront a mod NW
    const WalkArgsP ae = args_here(args);
    const uint32_t work = n_steps + n_visit / 2u;
    if (valid && ae->b.hrank[i] < 0) {
        const bool kick = ae->p.kick != 0;
        const double half_dt = ae->p.half_dt;
        const double ax = hax + lacc[0];
        const double ay = hay + lacc[1];
        const double az = haz + lacc[2];
        if (0 % NW == w) {
            ae->b.ax[i] = ax;
            if (kick) ae->b.vx[i] = ae->b.vx[i] + half_dt * ax;
        }
        if (1 % NW == w) {
            ae->b.ay[i] = ay;
            if (kick) ae->b.vy[i] = ae->b.vy[i] + half_dt * ay;
        }
        if (2 % NW == w) {
            ae->b.az[i] = az;
            if (kick) ae->b.vz[i] = ae->b.vz[i] + half_dt * az;
        }
    }
    // the group's work, the schedules' cost unit: the flushes' costs plus
    // half the visits (a visit measured half the time of a list step on
    // the 300k walk)
    if (valid && w == 0) ae->b.pcost[i] = work;
    if (tid == 0) {
        ae->mb.g_inter[g] = n_inter;
        ae->mb.g_visit[g] = n_visit;
        ae->mb.g_work[g] = work;
        ae->mb.g_t0[g] = t_start;
        ae->mb.g_t1[g] = wall_clock64();
        ae->mb.g_worker[g] = blockIdx.x * kWaves + (threadIdx.x >> 6);   // (w is 0 for a lone wavefront)
    }
    group_sync<NW>();   // the next group writes the exchanged sums and the list
    return work;
}

__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(3))) void k_walk_mixed(WalkArgs)
{
    const WalkArgsP args = (WalkArgsP)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(16))) unsigned char s_mem[kWaves * kWaveLds];
    __shared__ __attribute__((aligned(16))) uint32_t s_word[2][kWaves];
    __shared__ uint32_t s_take;
    const int w = static_cast<int>(uni(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    StepScalars* const sc = args->tb.sc;
    const uint32_t G = sc->n_groups;
    const uint32_t nblk = gridDim.x, waves = nblk * kWaves;
    const size_t tree_bytes = (static_cast<size_t>(sc->n_leaves) + sc->n_branch) * sizeof(MNode);
    // (19k bodies, 1.3 MB: walk 0.129 -> 0.122 ms; at 50k, 3.5 MB, +1%: there
    // the walk's own rounds overlap the misses)
    if (tree_bytes <= kWarmBytes / 2) warm_l2(args->mb.node, tree_bytes);
    // heaviest-first order pays while the tail decides the walk (few groups
    // per worker); with many groups per worker the key order's locality wins
    // (measured crossover between 8 and 33 groups per worker wave)
    const int sched = args->p.sched;
    const bool use_order = sched == 1 && G <= args->p.order_max_groups;
    // First the groups that are shared: order[0..C) in the cost order, the
    // list of k_mixed_nodes in key order; without a previous walk every group
    // of a small system (2 a block) and none of a larger one.  Every block's
    // first group is fixed by its place, and blocks ask the queue only after
    // that, so a system with fewer groups than blocks takes no atomic at all.
    // (With every take an atomic, 3,072 waves each closing eight queues on
    // one cache line held up the loads of the 561 waves that had a group for
    // 100 of the 336 us of a 19k walk.)
    uint32_t C = 0;
    bool listed = false;   // the shared groups come from a list, not 0..C-1
    if (sched != 2) {
        if (sc->work_prev == 0u) {
            C = G <= 2u * nblk ? G : 0u;
            listed = use_order;
        } else {
            C = min(use_order ? sc->n_coop : min(sc->n_big, kMaxShared), G);
            listed = true;
        }
    }
    uint32_t turn_no = 0;
    uint64_t work_done = 0;
    for (uint32_t k = blockIdx.x; k < C;) {
        uint32_t g = k;
        if (listed) {
            const WalkArgsP al = args_here(args);
            g = use_order ? al->mb.order[k] : al->mb.chunk[k];
        }
        g = uni(g);
        if (g < G) {
            const uint32_t work = walk_group<kWaves>(args, sc, g, w, lane, s_mem, s_word, turn_no);
            if (w == 0) work_done += work;
        }
        if (C <= nblk) break;   // every block had its only one
        if (threadIdx.x == 0) s_take = atomicAdd(&sc->queue[kQShared][0], 1u);
        __syncthreads();
        k = uni(nblk + s_take);
        __syncthreads();
    }
    __syncthreads();   // from here on every wavefront is on its own
    if (C < G) {
        unsigned char* const lds = s_mem + w * kWaveLds;
        uint32_t pos = 0, end = 0;   // the current chunk's groups (sched 2)
        uint32_t part = blockIdx.x % kWalkParts;   // key order: this XCD's runs first, then the other parts'
        // With no shared groups a wave's first group is fixed by its place too
        // (a block's waves take neighbouring places: they sit on the CU's four
        // SIMDs, so the costliest groups spread over the SIMDs); else the
        // queues serve the waves as their blocks finish.
        const uint32_t rank = blockIdx.x * kWaves + static_cast<uint32_t>(w);
        bool first_take = C == 0u;
        const uint32_t held = C == 0u ? waves : 0u;   // entries that are fixed
        auto take = [&](uint32_t row) {
            uint32_t q = 0;
            if (lane == 0) q = atomicAdd(&sc->queue[row][0], 1u);
            return uni(q);
        };
        auto held_part = [&](uint32_t x) { return C == 0u ? part_blocks(x, nblk) * kWaves : 0u; };
        for (;;) {
            uint32_t g;
            if (sched == 2) {
                // balanced chunks of consecutive groups, served by a dynamic queue;
                // every take consumes a chunk, so the loop ends after n_chunks takes
                while (pos >= end) {
                    const uint32_t q = first_take ? rank : held + take(kQOrder);
                    first_take = false;
                    const WalkArgsP ac = args_here(args);
                    if (q >= ac->p.n_chunks) break;
                    pos = uni(ac->mb.chunk[q]);
                    end = uni(ac->mb.chunk[q + 1]);
                }
                if (pos >= end) break;
                g = pos++;
            } else if (use_order) {
                // heaviest first from one queue: dealing the order out per XCD
                // measured 23% slower on the 300k walk (its span grows)
                const uint32_t q = C + (first_take ? rank : held + take(kQOrder));
                first_take = false;
                if (q >= G) break;
                g = args_here(args)->mb.order[q];
            } else {
                // key order, dealt out per XCD (5% shorter on the 300k walk, 4%
                // on a 32-system ensemble)
                uint32_t q;
                if (first_take) q = part_group(part, blockIdx.x / kWalkParts * kWaves + static_cast<uint32_t>(w));
                else q = part_group(part, held_part(part) + take(part));
                first_take = false;
                while (q >= G) {
                    // this part is closed: note it, learn which others are, and
                    // take from the next that may be open (a part once closed
                    // stays closed, so the loop ends).  Two atomics for a wave
                    // that leaves when all are; reading the queues' counters
                    // instead (relaxed loads, device scope) held up the last
                    // groups by 130 us at 300k.
                    uint32_t mask = 0;
                    if (lane == 0) mask = atomicOr(&sc->queue[kQClosed][0], 1u << part);
                    const uint32_t open = 0xffu & ~(uni(mask) | 1u << part);
                    if (open == 0u) break;
                    const uint32_t turned = ((open >> part) | (open << (kWalkParts - part))) & 0xffu;
                    part = (part + static_cast<uint32_t>(__builtin_ctz(turned))) % kWalkParts;
                    q = part_group(part, held_part(part) + take(part));
                }
                if (q >= G) break;
                g = q;
                if (C > 0u && args_here(args)->mb.gbig[g]) continue;   // walked by a block above
            }
            g = uni(g);
            if (g >= G) continue;   // a schedule entry outside the groups of this step
            work_done += walk_group<1>(args, sc, g, 0, lane, lds, s_word, turn_no);
        }
    }
    if (lane == 0 && work_done)
        atomicAdd(reinterpret_cast<unsigned long long*>(&sc->work_sum[blockIdx.x & 7u][0]), static_cast<unsigned long long>(work_done));
    // then the heavy bodies' chunk sums, in the walk's tail: a wave whose
    // groups are done takes work items while the last groups finish (its part
    // of the LDS holds the lane partials).  When the blocks with a group leave
    // enough waves, the items go to the last waves of the grid without a queue.
    const WalkArgsP at = args_here(args);
    const uint32_t items = at->p.heavy_items / kHeavyTogether;
    const HeavyArgs ha{at->b.px, at->b.py, at->b.pz, at->b.m, at->tb.sys, at->tb.n_sys, at->mb.hpart, at->p.soft2, at->p.G};
    const bool fixed = C == G && static_cast<uint64_t>(G) * kWaves + items <= waves;
    for (uint32_t k = 0;; ++k) {
        uint32_t q;
        if (fixed) {
            q = k == 0u ? waves - 1u - (blockIdx.x * kWaves + static_cast<uint32_t>(w)) : items;
        } else {
            q = 0;
            if (lane == 0) q = atomicAdd(&sc->queue[kQHeavy][0], 1u);
        }
        q = uni(q);
        if (q >= items) break;
        heavy_item(ha, q, lane, reinterpret_cast<double(*)[kHeavyRow]>(s_mem + w * kWaveLds));
    }
}

__global__ __launch_bounds__(kNT) void k_heavy_partial(Bodies b, TreeBuffers tb, MixedBuffers mb, MixedParams p)
{
    __shared__ double part[kWaves][3 * kHeavyTogether][kHeavyRow];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t waves = gridDim.x * kWaves;
    for (uint32_t item = blockIdx.x * kWaves + w; item < p.heavy_items / kHeavyTogether; item += waves)
        heavy_item(HeavyArgs{b.px, b.py, b.pz, b.m, tb.sys, tb.n_sys, mb.hpart, p.soft2, p.G}, item, lane, part[w]);
}

// One wavefront per (system, heavy rank, axis): lane l adds the chunk
// partials l, l + 64, ... (compensated), then the 64 lane sums are added in lane
// order -- a fixed order for a given system.
__global__ __launch_bounds__(kNT) void k_heavy_final(Bodies b, TreeBuffers tb, MixedBuffers mb, MixedParams p)
{
    __shared__ double lanes[kWaves][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t t = blockIdx.x * kWaves + w;
    const uint32_t a = t % 3, k = (t / 3) % kMaxHeavy, q = t / (3 * kMaxHeavy);
    if (q >= tb.n_sys) return;
    const SysScalars* sy = tb.sys + q;
    // the system's fields in one round (heavy_slot has kMaxHeavy entries)
    const uint32_t nh = sy->n_heavy, h = sy->heavy_slot[k], item0 = sy->heavy_item, nc = sy->heavy_chunks;
    if (k >= nh) return;
    double* accel = a == 0 ? b.ax : (a == 1 ? b.ay : b.az);
    double* vel = a == 0 ? b.vx : (a == 1 ? b.vy : b.vz);
    const double v_old = (p.kick && lane == 0) ? vel[h] : 0.0;   // loaded beside the partials
    ExactSum acc;
    const size_t first = item0 + static_cast<size_t>(k) * nc;
    // eight partials loaded per round before they are added (in chunk order)
    for (uint32_t c0 = static_cast<uint32_t>(lane); c0 < nc; c0 += 64 * 8) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t c = c0 + 64 * j;
            v[j] = c < nc ? mb.hpart[3 * (first + c) + a] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (c0 + 64 * j < nc) acc.add(v[j]);
    }
    lanes[w][lane] = acc.value();
    __builtin_amdgcn_wave_barrier();
    if (lane != 0) return;
    ExactSum tot;
    for (int l = 0; l < 64; ++l) tot.add(lanes[w][l]);
    const double v = tot.value();
    accel[h] = v;
    if (p.kick) vel[h] = v_old + p.half_dt * v;
}

// ------------------------------------------------------------ schedule
// Longest-processing-time order of the groups for the dynamic queue: groups
// go into 128 buckets of descending estimated cost (eight buckets per octave)
// and the queue serves the costliest bucket first.  The order inside a bucket
// is whatever the atomics give: it changes timing only, never results.
//
// Cost estimate, source 0: the previous step, i.e. the largest walk work of
// the groups any of the group's bodies were in (groups mostly persist from
// step to step).
// Source 1: the cost model, evaluated by k_group_features.
constexpr unsigned kSchedBlocks = 256;

// Cost estimate from the previous step: one wavefront per group takes the
// largest previous walk work of its bodies and counts the group in its
// block's bucket histogram, added to the step's counts.  The LEARNED form's
// estimate comes from k_group_features instead, which ends the same way.
__global__ __launch_bounds__(kNT) void k_sched_cost(size_t n, Bodies b, TreeBuffers tb, MixedBuffers mb,
                                                    uint32_t max_groups)
{
    __shared__ uint32_t hist[kSchedBuckets];
    const uint32_t G = tb.sc->n_groups;
    if (G > max_groups) return;   // the walk will not use an order this step
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < kSchedBuckets) hist[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t waves = gridDim.x * kWaves;
    for (uint32_t g = blockIdx.x * kWaves + (threadIdx.x >> 6); g < G; g += waves) {
        const uint32_t i0 = mb.gfirst[g], cnt = mb.gfirst[g + 1] - i0;
        uint32_t m = static_cast<uint32_t>(lane) < cnt ? b.pcost[i0 + lane] : 0u;
        for (int o = 32; o > 0; o >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o, 64)));
        if (lane == 0) {
            mb.gcost[g] = static_cast<float>(m);
            atomicAdd(&hist[cost_bucket(static_cast<float>(m))], 1u);
        }
    }
    sched_hist_add(tb, hist);
}

// Every block scans the step's bucket counts into the buckets' first places,
// then places tiles of 256 groups: LDS counters rank a tile's groups inside
// their buckets, one global atomic per bucket reserves the tile's range.
__global__ __launch_bounds__(kNT) void k_sched_scatter(size_t n, TreeBuffers tb, MixedBuffers mb, uint32_t max_groups)
{
    static_assert(kSchedBuckets == 128 && kNT >= 128, "two waves scan the bucket counts");
    __shared__ uint32_t cnt[kSchedBuckets];
    __shared__ uint32_t base[kSchedBuckets];
    __shared__ uint32_t first[kSchedBuckets];
    __shared__ uint32_t wave0_total;
    const uint32_t G = tb.sc->n_groups;
    if (G > max_groups) return;
    if (threadIdx.x < kSchedBuckets) {
        uint32_t v = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) v += tb.sc->sched_hist[c][threadIdx.x];
        const uint32_t incl = wave_incl_scan(v);
        if (threadIdx.x == 63) wave0_total = incl;
        first[threadIdx.x] = incl - v;
    }
    __syncthreads();
    if (threadIdx.x >= 64 && threadIdx.x < kSchedBuckets) first[threadIdx.x] += wave0_total;
    if (blockIdx.x == 0) {
        // the groups of the buckets above the sharing limit come first
        __syncthreads();
        if (threadIdx.x == 0 && tb.sc->work_prev != 0u)
            tb.sc->n_coop = first[cost_bucket(static_cast<float>(share_limit(tb.sc, mb.walk_waves)))];
    }
    for (uint32_t t0 = blockIdx.x * kNT; t0 < G; t0 += gridDim.x * kNT) {
        if (threadIdx.x < kSchedBuckets) cnt[threadIdx.x] = 0;
        __syncthreads();
        const uint32_t g = t0 + threadIdx.x;
        uint32_t bk = 0, local = 0;
        if (g < G) {
            bk = cost_bucket(mb.gcost[g]);
            local = atomicAdd(&cnt[bk], 1u);
        }
        __syncthreads();
        if (threadIdx.x < kSchedBuckets && cnt[threadIdx.x])
            base[threadIdx.x] = first[threadIdx.x] + atomicAdd(&tb.sc->sched_cursor[threadIdx.x], cnt[threadIdx.x]);
        __syncthreads();
        if (g < G) mb.order[base[bk] + local] = g;
        __syncthreads();
    }
}

// Split schedule.  Group weights: the estimated cost in units of 8 list
// entries, plus one (so empty estimates still count), at most 65535.
// Entries from n_groups to n are zero, so a scan over n adds the groups only.
__global__ __launch_bounds__(kNT) void k_chunk_weights(size_t n, TreeBuffers tb, MixedBuffers mb,
                                                       uint32_t* __restrict__ w)
{
    const size_t g = static_cast<size_t>(blockIdx.x) * kNT + threadIdx.x;
    if (g >= n) return;
    if (g >= tb.sc->n_groups) {
        w[g] = 0;
        return;
    }
    const float c = fmaxf(mb.gcost[g], 0.f) * 0.125f + 1.f;
    w[g] = c >= 65535.f ? 65535u : static_cast<uint32_t>(c);
}

// chunk[c] = first group whose exclusive weight prefix reaches c / C of the
// total, so chunk c covers the groups whose weight starts in its C-th of the
// total; chunk[0] = 0, chunk[C] = G.
__global__ __launch_bounds__(kNT) void k_chunk_bounds(TreeBuffers tb, MixedBuffers mb,
                                                      const uint32_t* __restrict__ prefix, uint32_t n_chunks)
{
    const uint32_t c = blockIdx.x * kNT + threadIdx.x;
    if (c > n_chunks) return;
    const uint32_t G = tb.sc->n_groups;
    if (c == 0 || c == n_chunks) {
        mb.chunk[c] = c == 0 ? 0u : G;
        return;
    }
    const uint64_t target = static_cast<uint64_t>(c) * tb.sc->cost_total / n_chunks;
    uint32_t lo = 0, len = G;   // first g with prefix[g] >= target
    while (len > 0) {
        const uint32_t half = len >> 1;
        if (prefix[lo + half] < target) {
            lo += half + 1;
            len -= half + 1;
        } else {
            len = half;
        }
    }
    mb.chunk[c] = lo;
}

inline unsigned nblk(size_t n) { return static_cast<unsigned>((n + kNT - 1) / kNT > 0 ? (n + kNT - 1) / kNT : 1); }

}  // namespace

void launch_chunks(const Bodies& b, size_t n, const TreeBuffers& tb, const MixedBuffers& mb, int source,
                   uint32_t n_chunks, hipStream_t s)
{
    if (source == 0) k_sched_cost<<<kSchedBlocks, kNT, 0, s>>>(n, b, tb, mb, 0xffffffffu);   // previous walk work
    // weights into mb.order, their exclusive prefix into mb.base (both free
    // once the node array is built)
    k_chunk_weights<<<nblk(n), kNT, 0, s>>>(n, tb, mb, mb.order);
    scan_exclusive_u32(mb.order, mb.base, &tb.sc->cost_total, n, tb.scan_tmp, s);
    k_chunk_bounds<<<(n_chunks + kNT) / kNT, kNT, 0, s>>>(tb, mb, mb.base, n_chunks);
}

void launch_mixed_layout(size_t n, TreeBuffers& tb, MixedBuffers& mb, const GroupParams& gp, hipStream_t s)
{
    const unsigned hg = hist_blocks(n);
    k_split_hist<<<std::max(hg, nblk(n)), kNT, 0, s>>>(n, tb, hg);
    scan_tile_offsets(tb.scan_tmp, n, s);
    k_slots<<<nblk(n), kNT, 0, s>>>(n, tb, mb, gp);
}

void launch_mixed_groups(const Bodies& b, size_t n, TreeBuffers& tb, MixedBuffers& mb, const GroupParams& gp,
                         double G, hipStream_t s)
{
    k_group_marks<<<nblk(2 * n), kNT, 0, s>>>(n, tb, mb, gp.gmax < 1 ? 1u : (gp.gmax > 64 ? 64u : gp.gmax));
    // group index of every first body: the group flags scanned, the tile
    // sums counted by k_group_marks, the block-local scan in k_mixed_nodes
    scan_tile_offsets(tb.gtile, n, s);
    k_mixed_nodes<<<nblk(2 * n), kNT, 0, s>>>(n, b, tb, mb, G);
}

unsigned mixed_walk_blocks(int device)
{
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k_walk_mixed), kNT, 0) !=
            hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    return static_cast<unsigned>(cus * per_cu);
}

void launch_schedule(const Bodies& b, size_t n, const TreeBuffers& tb, const MixedBuffers& mb, int source,
                     uint32_t max_groups, hipStream_t s)
{
    // source 1: k_group_features has already estimated and counted the groups
    if (source == 0) k_sched_cost<<<kSchedBlocks, kNT, 0, s>>>(n, b, tb, mb, max_groups);
    k_sched_scatter<<<kSchedBlocks, kNT, 0, s>>>(n, tb, mb, max_groups);
}

void launch_walk_mixed(const Bodies& b, size_t n, const TreeBuffers& tb, const MixedBuffers& mb,
                       const MixedParams& p, unsigned blocks, hipStream_t s)
{
    if (n == 0 || blocks == 0) return;
    k_walk_mixed<<<blocks, kNT, 0, s>>>(WalkArgs{b, tb, mb, p});
}

void launch_heavy_direct(const Bodies& b, const TreeBuffers& tb, const MixedBuffers& mb, const MixedParams& p,
                         bool in_walk, hipStream_t s)
{
    if (p.heavy_items == 0) return;
    const unsigned hb = std::min<unsigned>((p.heavy_items / kHeavyTogether + kWaves - 1) / kWaves, 4096u);
    if (!in_walk) k_heavy_partial<<<hb, kNT, 0, s>>>(b, tb, mb, p);
    k_heavy_final<<<(tb.n_sys * 3 * kMaxHeavy + kWaves - 1) / kWaves, kNT, 0, s>>>(b, tb, mb, p);
}

}  // namespace bh
