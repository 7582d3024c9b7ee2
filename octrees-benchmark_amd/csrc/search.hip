// H5: radius searches (neighbors / neighborsPrune / neighborsStruct x sphere / circle / cube /
// square) on gfx950.
//
// Two kernels, both giving exactly the reference's results for every query:
//  - k_group: a group of 8 lanes per query, each group with its own traversal (result lists, and counts
//    of queries that are far apart or few);
//  - k_count: 16 - 64 consecutive queries per wave that share one traversal (counts of many queries that
//    lie together, the all-points searches; k_lists: their result lists). FP32 sphere counts test leaves on
//    the matrix cores and judge children by tight boxes.
//
// Per-point tests:
//  - FP64: the reference's isInside expression (kernel_3d.hpp:127-138, 232-242; kernel_2d.hpp:53-63,
//    153-162), evaluated as written (no contraction).
//  - FP32_RECHECK (sphere, circle): leaf-recentred FP32 coordinates a (w = |a|^2 precomputed) and
//    b = fl32(q - c_leaf); t = fma(ax, -2bx, fma(ay, -2by, fma(az, -2bz, w + C))) (circle: fma(ax,
//    ax - 2bx, fma(ay, ay - 2by, C))) approximates |p - q|^2 - R + hw with a band hw = 2^-18 (amax +
//    |b|^2 + R), amax = max |a|^2 over the leaf, that covers every rounding of this evaluation and of the
//    reference's FP64 one (its bound: see the leaf's tests in k_count). A set sign bit is inside, t > 2 hw
//    outside, and what lies between is decided by the FP64 expression.
//  - A leaf/query pair whose FP32 terms could overflow or become denormal (fp32_range), or a leaf holding a
//    non-finite FP32 point (then amax = inf), is decided in FP64 throughout.
//  - Cube/square tests are comparisons only and run on the FP64 coordinates in both modes.
#include <algorithm>
#include <type_traits>

#include "grid.hpp"
#include "search_common.hpp"

namespace oct {

// ------------------------------------------------------------------ group kernel: one query per 8 lanes
// Result lists, and counts of queries that lie far apart. A group of 8 lanes walks its own query's
// traversal; a wave serves 8 queries, each with its own position in the tree:
//  - a popped node's 8 children are judged one per lane with the reference's FP64 expressions, 8 nodes
//    (one per group) per step. The children still to be visited are one bit per (level, lane): lane c's
//    `pend` has bit L set while child c at level L waits, `lvl` has bit L set while any does. Taking the
//    highest waiting octant of the deepest level is the reference's LIFO order (singleTraversal,
//    linear_octree.hpp:653-686), so lists come out in the reference's emission order;
//  - the OVERLAP leaves (and, when lists are filled, the INSIDE ranges) of a popped node go to the
//    group's queue in octant order, with the leaf's FP32 terms formed by the lane that judged it. When
//    no group can go on (queue full or traversal done), every group tests its queued points, 16 per
//    step, and writes its hits side by side: 8 lanes' hits of a step are consecutive list entries.
// What bounds it: vector issue (4.2 k vector instructions per wave of 8 queries at 84 neighbours each)
// and, for few queries, the chain of dependent loads of one traversal. Against a wave of 64 queries that
// shares one traversal, each lane writing its own list and reading the points one by one: 10 000 random
// centres of a 1 M-point box, r = 2.5 (both list passes) 14.6 -> 0.45 ms; 1 M consecutive points of a
// 5 M-point tile, r = 1, index lists 2.91 -> 2.14 ms; 2 M of 20 M, r = 2.5, ranges 17.2 -> 12.1 ms.
constexpr int kGroupLanes = 8;
constexpr int kGroupsPerWave = 64 / kGroupLanes;
constexpr int kGroupQueue = 16;  // queued items per group; a pop adds at most 8
constexpr int kGroupMaxLevels = (int)kMaxDepth;  // levels that can hold internal nodes (0 .. 20)

// A queued item, [slot * 8 + group]: the point range (bit 31 of last: an INSIDE range) and, for an FP32
// leaf, its terms. One slot more than can be filled: groups that are done read it while others go on.
template <bool FP32>
struct GroupItems {
    uint2 range[(kGroupQueue + 1) * kGroupsPerWave];
};
template <>
struct GroupItems<true> {
    uint4 range_xy[(kGroupQueue + 1) * kGroupsPerWave];  // first, last, -2bx, -2by (bits)
    uint4 z_c_lim[(kGroupQueue + 1) * kGroupsPerWave];   // -2bz, C, lim (bits)
};

// boxIntersect / boxOverlap of one node without branches: in = INSIDE, ov = OVERLAP (neither: OUTSIDE).
// The comparisons and sums are classify64's and overlap64's, in the same order.
template <int KERNEL, int ALGO>
__device__ inline void judge_node(const Query &q, const NodeRec &n, double rx, double ry, double rz, bool &in, bool &ov) {
    constexpr bool is3d = KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CUBE;
    if (ALGO == OCT_ALGO_NEIGHBORS || KERNEL == OCT_KERNEL_CUBE || KERNEL == OCT_KERNEL_SQUARE) {
        const double hx = n.cx + rx, lx = n.cx - rx, hy = n.cy + ry, ly = n.cy - ry, hz = n.cz + rz, lz = n.cz - rz;
        bool out = (hx < q.lox) | (hy < q.loy) | (lx > q.hix) | (ly > q.hiy);
        if (is3d) out |= (hz < q.loz) | (lz > q.hiz);
        bool inside = false;
        if (ALGO != OCT_ALGO_NEIGHBORS) {
            inside = (hx <= q.hix) & (hy <= q.hiy) & (lx >= q.lox) & (ly >= q.loy);
            if (is3d) inside &= (hz <= q.hiz) & (lz >= q.loz);
        }
        in = !out & inside;
        ov = !out & !inside;
    } else {
        const double dx = fabs(q.x - n.cx), dy = fabs(q.y - n.cy), dz = is3d ? fabs(q.z - n.cz) : 0.0;
        bool out = (dx > q.r + rx) | (dy > q.r + ry);
        if (is3d) out |= dz > q.r + rz;
        const double ex = dx + rx, ey = dy + ry;
        const double fx = dmax0(dx - rx), fy = dmax0(dy - ry);
        double smax = ex * ex + ey * ey, smin = fx * fx + fy * fy;
        const bool nx = dx < rx, ny = dy < ry;
        bool two = nx & ny;  // at least two axes within the node's slab (the two of a 2-D kernel)
        if (is3d) {
            const double ez = dz + rz, fz = dmax0(dz - rz);
            smax = smax + ez * ez, smin = smin + fz * fz;
            two |= (dz < rz) & (nx | ny);
        }
        const bool inside = smax <= q.R;
        in = !out & inside;
        ov = !out & !inside & (two | (smin <= q.R));
    }
}

// One wave's queries (tile: 8 slots). MODE 0: neighbour counts; 1: counts and list-entry counts; 2: fill the
// lists at their offsets. root and s_rad (level radii): the slots' cloud; limit: the first slot past its
// valid ones.
template <int KERNEL, int ALGO, int PREC, int MODE, class Items>
__device__ __attribute__((always_inline)) inline void group_tile(const SearchArgs &a, const uint32_t tile, const uint32_t root,
                                                                 const uint32_t limit, Items &Q, const double *s_rad,
                                                                 uint32_t *s_gc) {
    constexpr bool kFp32 = PREC == OCT_PREC_FP32_RECHECK && (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE);
    constexpr bool kRanges = ALGO == OCT_ALGO_STRUCT || ALGO == OCT_ALGO_APPROX;  // lists of [first, last) ranges
    constexpr uint32_t kInside = 0x80000000u;
    constexpr uint64_t kBit0 = 0x0101010101010101ull;  // the first lane of every group
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t grp = lane >> 3, c = lane & 7u, gshift = lane & 56u;
    const uint32_t below = (1u << c) - 1u;
    const uint32_t slot = tile * kGroupsPerWave + grp;
    const bool valid = slot < limit;
    auto wsync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto group_bits = [&](bool p) -> uint32_t { return (uint32_t)(ballot64(p) >> gshift) & 255u; };

    Query q;
    uint32_t qid = 0;
    q.x = q.y = q.z = 0.0;
    q.r = 0.0;
    if (valid) {
        qid = a.order ? a.order[slot] : slot;
        if (a.qxyz) {
            q.x = a.qxyz[3 * (size_t)qid], q.y = a.qxyz[3 * (size_t)qid + 1], q.z = a.qxyz[3 * (size_t)qid + 2];
        } else {
            const double4 p = a.p64[a.qidx ? a.qidx[qid] : qid];
            q.x = p.x, q.y = p.y, q.z = p.z;
        }
        q.r = a.qrad ? a.qrad[qid] : a.radius;
    }
    q.R = q.r * q.r;
    q.lox = q.x - q.r, q.loy = q.y - q.r, q.loz = q.z - q.r;
    q.hix = q.x + q.r, q.hiy = q.y + q.r, q.hiz = q.z + q.r;
    if (KERNEL == OCT_KERNEL_CUBE || KERNEL == OCT_KERNEL_SQUARE) box_radii(a, valid, qid, q);
    const float qRf = (float)q.R;
    uint32_t *out = nullptr;  // MODE 2: the query's list
    if (MODE == 2 && valid) out = a.entries + a.offsets[qid] * (kRanges ? 2u : 1u);

    uint32_t cnt = 0, ecnt = 0;  // MODE 0, 1: this lane's share of the query's counts
    uint32_t off = 0;            // MODE 2: entries written so far (the same in the group's lanes)
    uint32_t n_class = 0, n_recheck = 0, n_csteps = 0, n_tsteps = 0;
    uint64_t n_test = 0;
    uint32_t qn = 0;             // queued items
    uint32_t lvl = 0, pend = 0;  // levels with waiting children; levels at which this lane's child waits
    bool overflow = false;

    // a judged child of the query's traversal is counted, queued, made to wait or dropped. Called by all
    // lanes of a group at once (act = false: no child in this lane); L is the child's level.
    auto take = [&](const bool act, const NodeRec &nr, const uint32_t gc, const float am, const uint32_t L) {
        bool in, ov;
        judge_node<KERNEL, ALGO>(q, nr, s_rad[3 * L], s_rad[3 * L + 1], s_rad[3 * L + 2], in, ov);
        // neighborsApprox beyond its precision level: the node's range whole, or nothing (linear_octree.hpp:987-994)
        if (ALGO == OCT_ALGO_APPROX && L > a.approx_level) in = a.approx_upper != 0, ov = false;
        in &= act, ov &= act;
        n_class += act ? 1u : 0u;
        const bool some = nr.last > nr.first;
        const bool leaf = ov & (gc == 0) & some;  // an empty leaf adds nothing
        if (MODE != 2 && in) {
            cnt += nr.last - nr.first;
            if (kRanges) ecnt++;  // NeighborSet::addRange keeps empty ranges (neighbor_set.hpp:84-89)
        }
        const bool item = leaf | (MODE == 2 && in && (kRanges || some));
        const uint32_t im = group_bits(item);
        if (item) {
            const uint32_t s = (qn + (uint32_t)__popc(im & below)) * kGroupsPerWave + grp;
            const uint32_t last = nr.last | (MODE == 2 && in ? kInside : 0u);
            if (leaf) n_test += nr.last - nr.first;
            if constexpr (kFp32) {
                // the leaf's FP32 form with the band folded in: t = w + C - 2 a.b (circle: its two axes)
                // approximates |p - q|^2 - R + hw; its bound stands at the count kernel's leaf tests. Sign
                // bit set: inside; bits above lim: outside; else (or lim = ~0, where the FP32 terms could
                // overflow or become denormal) the FP64 test decides.
                const float bx = (float)(q.x - nr.cx), by = (float)(q.y - nr.cy), bz = (float)(q.z - nr.cz);
                const float b2 = KERNEL == OCT_KERNEL_SPHERE ? __builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz))
                                                             : __builtin_fmaf(bx, bx, by * by);
                const float sum = (am + b2) + qRf;
                const float hw = 3.814697265625e-06f * sum;  // 2^-18
                Q.range_xy[s] = make_uint4(nr.first, last, __float_as_uint(-2.0f * bx), __float_as_uint(-2.0f * by));
                Q.z_c_lim[s] = make_uint4(__float_as_uint(-2.0f * bz), __float_as_uint((hw - qRf) + b2),
                                          fp32_range(sum) ? __float_as_uint(2.0f * hw) : 0xffffffffu, 0u);
            } else {
                Q.range[s] = make_uint2(nr.first, last);
            }
        }
        qn += (uint32_t)__popc(im);
        const bool wait = ov & (gc != 0);
        const uint64_t wm = ballot64(wait);
        if (wm) {
            if (wait) s_gc[L * 64 + lane] = gc, pend |= 1u << L;
            if ((wm >> gshift) & 255u) lvl |= 1u << L;
        }
    };

    // tests the queued points of every group, 16 per step, in queue order
    auto flush = [&]() {
        wsync();
        uint32_t it = 0, i = 0;
        bool fresh = true;     // step starts a new item
        uint64_t carry = 0;    // range lists: groups (bit 8g) whose current run reaches the step's first point
        while (ballot64(it < qn)) {
            n_tsteps++;
            const uint32_t s = it * kGroupsPerWave + grp;
            uint32_t first, last, lim = 0;
            float ux = 0.f, uy = 0.f, uz = 0.f, C = 0.f;
            if constexpr (kFp32) {
                const uint4 A = Q.range_xy[s], B = Q.z_c_lim[s];
                first = A.x, last = A.y, ux = __uint_as_float(A.z), uy = __uint_as_float(A.w);
                uz = __uint_as_float(B.x), C = __uint_as_float(B.y), lim = B.z;
            } else {
                const uint2 A = Q.range[s];
                first = A.x, last = A.y;
            }
            const bool ins = MODE == 2 && (last & kInside) != 0;
            const uint32_t e = MODE == 2 ? last & ~kInside : last;
            if (fresh) i = first;
            const uint32_t rem = it < qn ? e - i : 0u;
            const uint32_t i0 = i + c, i1 = i0 + 8;
            const bool v0 = c < rem, v1 = c + 8 < rem;
            bool in0 = false, in1 = false;
            if (v0 & !ins) {  // reads up to 15 points past the range: the sorted clouds are padded (kPointPad)
                if constexpr (kFp32) {
                    const float4 p0 = a.p32[i0], p1 = a.p32[i1];
                    float t0, t1;
                    if (KERNEL == OCT_KERNEL_SPHERE) {
                        t0 = __builtin_fmaf(p0.x, ux, __builtin_fmaf(p0.y, uy, __builtin_fmaf(p0.z, uz, p0.w + C)));
                        t1 = __builtin_fmaf(p1.x, ux, __builtin_fmaf(p1.y, uy, __builtin_fmaf(p1.z, uz, p1.w + C)));
                    } else {
                        t0 = __builtin_fmaf(p0.x, p0.x + ux, __builtin_fmaf(p0.y, p0.y + uy, C));
                        t1 = __builtin_fmaf(p1.x, p1.x + ux, __builtin_fmaf(p1.y, p1.y + uy, C));
                    }
                    const uint32_t d0 = __float_as_uint(t0), d1 = __float_as_uint(t1);
                    in0 = (int32_t)d0 < 0, in1 = v1 & ((int32_t)d1 < 0);
                    const bool k0 = d0 <= lim, k1 = v1 & (d1 <= lim);
                    if (k0 | k1) {
                        if (k0) {
                            const double4 pd = a.p64[i0];
                            in0 = inside64<KERNEL>(q, pd.x, pd.y, pd.z);
                            n_recheck++;
                        }
                        if (k1) {
                            const double4 pd = a.p64[i1];
                            in1 = inside64<KERNEL>(q, pd.x, pd.y, pd.z);
                            n_recheck++;
                        }
                    }
                } else {
                    const double4 p0 = a.p64[i0], p1 = a.p64[i1];
                    in0 = inside64<KERNEL>(q, p0.x, p0.y, p0.z);
                    in1 = v1 & inside64<KERNEL>(q, p1.x, p1.y, p1.z);
                }
            }
            if (MODE == 2 && ins) in0 = v0, in1 = v1;
            const bool next = rem <= 16;  // the item ends with this step
            if (MODE != 2) cnt += in0 ? 1u : 0u, cnt += in1 ? 1u : 0u;
            if constexpr (kRanges && MODE != 0) {
                // runs as lane masks: a hit starts one when the point before it is none, a miss ends one
                const bool one = MODE == 2 && ins;  // an INSIDE range is one entry, written below
                const uint64_t m0 = ballot64(in0 & !one), m1 = ballot64(in1 & !one);
                const uint64_t pr0 = ((m0 << 1) & ~kBit0) | carry, pr1 = ((m1 << 1) & ~kBit0) | ((m0 >> 7) & kBit0);
                const uint64_t st0 = m0 & ~pr0, st1 = m1 & ~pr1;
                if (MODE == 1) {
                    ecnt += __builtin_amdgcn_inverse_ballot_w64(st0) ? 1u : 0u;
                    ecnt += __builtin_amdgcn_inverse_ballot_w64(st1) ? 1u : 0u;
                } else {
                    const uint32_t sb = ((uint32_t)(st0 >> gshift) & 255u) | (((uint32_t)(st1 >> gshift) & 255u) << 8);
                    const uint32_t r0 = off + (uint32_t)__popc(sb & below), r1 = off + (uint32_t)__popc(sb & ((1u << (c + 8)) - 1u));
                    off += (uint32_t)__popc(sb);
                    if (__builtin_amdgcn_inverse_ballot_w64(st0)) out[2 * (size_t)r0] = i0;
                    if (__builtin_amdgcn_inverse_ballot_w64(st1)) out[2 * (size_t)r1] = i1;
                    if (__builtin_amdgcn_inverse_ballot_w64(~m0 & pr0)) out[2 * (size_t)r0 - 1] = i0;
                    if (__builtin_amdgcn_inverse_ballot_w64(~m1 & pr1)) out[2 * (size_t)r1 - 1] = i1;
                    // the leaf ends with the step's last point and that is a hit
                    if (in1 & !one & (c == 7) & (rem == 16)) out[2 * (size_t)off - 1] = e;
                    if (one && it < qn) {
                        if (c == 0) out[2 * (size_t)off] = first, out[2 * (size_t)off + 1] = e;
                        off++;
                    }
                }
                carry = (m1 >> 7) & kBit0 & ~ballot64(next);
            } else if constexpr (MODE == 2) {
                const uint32_t m = group_bits(in0) | (group_bits(in1) << 8);
                if (in0) out[off + (uint32_t)__popc(m & below)] = i0;
                if (in1) out[off + (uint32_t)__popc(m & ((1u << (c + 8)) - 1u))] = i1;
                off += (uint32_t)__popc(m);
            }
            const bool done = next | (kRanges && ins);
            fresh = done;
            i += 16;
            if (it < qn && done) it++;
        }
        wsync();  // the queue is rewritten next
        qn = 0;
    };

    // root (singleTraversal, linear_octree.hpp:655-662): judged by the group's first lane
    take(valid && c == 0, a.nodes[root], a.child[root], a.amax[root], 0);
    for (;;) {
        for (;;) {
            const bool go = lvl != 0 && qn <= (uint32_t)(kGroupQueue - 8);
            if (!ballot64(go)) break;
            n_csteps++;
            if (go) {
                wsync();
                const uint32_t L = 31u - (uint32_t)__clz(lvl);  // the deepest level with waiting children
                const uint32_t wm = group_bits((pend >> L) & 1u);
                const uint32_t oct = 31u - (uint32_t)__clz(wm);  // the last one made to wait
                const uint32_t fc = s_gc[L * 64 + gshift + oct];
                if (c == oct) pend &= ~(1u << L);
                if ((wm & (wm - 1u)) == 0) lvl &= ~(1u << L);
                const uint32_t node = fc + c;
                const NodeRec nr = a.nodes[node];
                const uint32_t gc = a.child[node];
                const float am = kFp32 ? a.amax[node] : 0.0f;  // (an internal node's value is not used)
                const bool fits = L + 1 < a.levels || gc == 0;
                overflow |= !fits;  // an internal node below the tree's last level: cannot happen
                take(fits, nr, gc, am, L + 1);
            }
        }
        if (!ballot64(qn != 0)) break;  // nothing queued: every traversal is done
        flush();
    }

    if (ballot64(overflow) && lane == 0) atomicOr(a.err, kErrStack);
    if (MODE != 2) {
        cnt += lane_xor<1>(cnt), cnt += lane_xor<2>(cnt), cnt += lane_xor<4>(cnt);
        if (MODE == 1 && kRanges) ecnt += lane_xor<1>(ecnt), ecnt += lane_xor<2>(ecnt), ecnt += lane_xor<4>(ecnt);
        if (MODE == 1 && !kRanges) ecnt = cnt;  // index lists: one entry per neighbour
        if (valid && c == 0) {
            if (a.counts) a.counts[qid] = cnt;
            if (MODE == 1 && a.ecounts) a.ecounts[qid] = ecnt;
            if (MODE == 1 && a.ecounts64) a.ecounts64[qid] = ecnt;
        }
    }
    if (a.stats) {
        uint64_t nb = (valid && c == 0) ? cnt : 0, nc = n_class, nr = n_recheck;
        for (int o = 32; o > 0; o >>= 1) {
            nc += __shfl_xor(nc, o), n_test += __shfl_xor(n_test, o);
            nr += __shfl_xor(nr, o), nb += __shfl_xor(nb, o);
        }
        if (lane == 0) {
            atomicAdd(&a.stats[0], (unsigned long long)nc);
            atomicAdd(&a.stats[1], (unsigned long long)n_test);
            if (nr) atomicAdd(&a.stats[2], (unsigned long long)nr);
            atomicAdd(&a.stats[3], (unsigned long long)nb);
            atomicAdd(&a.stats[4], 64ull * n_csteps);
            atomicAdd(&a.stats[5], 128ull * n_tsteps);
        }
    }
}

template <int PREC, int KERNEL>
constexpr bool group_fp32() {
    return PREC == OCT_PREC_FP32_RECHECK && (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE);
}

template <int KERNEL, int ALGO, int PREC, int MODE>
__global__ __launch_bounds__(kSearchBlock) void k_group(const SearchArgs a, const uint32_t block0) {
    __shared__ GroupItems<group_fp32<PREC, KERNEL>()> s_items[kWaves];
    __shared__ double s_rad[3 * (kMaxDepth + 1)];
    extern __shared__ uint32_t s_gc_all[];  // per wave, per level: each lane's child's first child
    for (uint32_t i = threadIdx.x; i < 3 * (kMaxDepth + 1); i += kSearchBlock) s_rad[i] = a.radtab[i];
    __syncthreads();
    const uint32_t w = threadIdx.x >> 6, tile = (block0 + blockIdx.x) * kWaves + w;
    if (uniform_u32(tile * kGroupsPerWave) >= a.nq) return;
    group_tile<KERNEL, ALGO, PREC, MODE>(a, tile, 0u, a.nq, s_items[w], s_rad, s_gc_all + (size_t)w * a.levels * 64);
}

// Counts over a forest (batches): resident waves take eighths of the 64-slot wave tiles, each of one cloud,
// from a counter until the device-resident number of tiles has been served.
// Forms chosen as for one cloud (shared_counts). 48 clouds of 12 M points together, sparse queries:
// k_count_queue 2.65 ms, this one 0.55.
template <int KERNEL, int ALGO, int PREC>
__global__ __launch_bounds__(kSearchBlock) void k_group_queue(const SearchArgs a) {
    __shared__ GroupItems<group_fp32<PREC, KERNEL>()> s_items[kWaves];
    __shared__ double s_rad[kWaves][3 * (kMaxDepth + 1)];
    extern __shared__ uint32_t s_gc_all[];
    constexpr uint32_t kParts = 64 / kGroupsPerWave;
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t nparts = uniform_u32(*a.queue_tiles) * kParts;
    for (;;) {
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(a.queue_next, 1u);
        t = readlane_u32(t, 0);
        if (t >= nparts) return;
        const uint32_t ti = uniform_u32(a.tile_info[t / kParts]);
        const uint32_t cloud = ti & 0xfffffu, limit = (t / kParts) * 64 + (ti >> 20);
        if (t * kGroupsPerWave >= limit) continue;
        for (uint32_t i = lane; i < 3 * (kMaxDepth + 1); i += 64) s_rad[w][i] = a.radtab[66 * (size_t)cloud + i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        group_tile<KERNEL, ALGO, PREC, 0>(a, t, uniform_u32(a.roots[cloud]), min(limit, a.nq), s_items[w], s_rad[w],
                                          s_gc_all + (size_t)w * a.levels * 64);
    }
}

// ------------------------------------------------------------------ count-mode kernel
// Per-query neighbour counts only (the harness keeps result.size(), neighbor_benchmarks.hpp:509).
// G queries per wave, S = 64 / G lanes per query: lane = g * G + j serves query j with "group" g.
//  - the 8 children of a popped node are judged together from per-axis terms (judge8 below);
//  - a leaf's points are staged once per wave in LDS and split across the S lanes of each query
//    (lane group g takes points g, g + S, ...); each staged chunk is padded with sentinel points
//    that are never inside and never in the FP32 band, so every lane runs the same 4x-unrolled
//    trip count with immediate LDS offsets; partial counts are summed at the end;
//  - a smaller G shrinks the union of the wave's traversals (fewer masked-off lane slots), a
//    larger one shares each judgement of 8 children among fewer lanes.
// Empty leaves are skipped: they add nothing to a count whatever their class. Counts do not
// depend on the order of the traversal, which is therefore free.

// Occupancy targets (waves per SIMD), measured on the 50 M-point tile for the sphere kernel with the
// Struct / Prune algorithms: 7 for FP32 (72 VGPRs, 12 bytes of scratch touched at a wave's start and end; at 8
// the 64-VGPR and 72-SGPR budget spilled the children's judgement masks and the search ran 3 % slower), 6 for
// FP64 (80 VGPRs). The other variants keep the compiler's choice (forcing them spills registers).
template <int KERNEL, int ALGO, int PREC>
constexpr int count_waves() {
    if (ALGO == OCT_ALGO_NEIGHBORS || !(KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE)) return 2;
    return PREC == OCT_PREC_FP32_RECHECK ? 7 : 6;
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// leaf_mfma's terms of the queries that want the leaf, compacted
struct MfmaQueries {
    struct alignas(16) Lim {
        uint32_t lim, home;  // band limit (float bits), lane
        __device__ void operator=(const uint2 &v) { lim = v.x, home = v.y; }
    };
    float4 u[64];  // -2 b, 1
    float4 c[64];  // C four times: the accumulator the products are added to
    Lim lh[64];    // 1 KB after c
    alignas(16) uint32_t acc[64];
};
// One wave tile (G queries) of a search, run by one wave. MODE 0: neighbour counts. MODE 1 (range lists,
// G = 64): counts and list-entry counts. MODE 2 (G = 64): the lists, in the reference's emission order.
template <int KERNEL, int ALGO, int PREC, int G, bool STATS, int MODE = 0>
__device__ __attribute__((always_inline)) inline void count_tile(const SearchArgs &a, const uint32_t tile) {
    constexpr int S = 64 / G;
    static_assert(MODE == 0 || G == 64, "lists: one lane per query");
    constexpr bool kRanges = ALGO == OCT_ALGO_STRUCT || ALGO == OCT_ALGO_APPROX;  // lists of [first, last) ranges
    constexpr bool kFp32 = PREC == OCT_PREC_FP32_RECHECK && (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE);
    // real points per staging chunk: 64 FP32 or 48 FP64 points (leaves average ~30 points; a small
    // chunk keeps the LDS per block low enough for 7 (FP32) or 6 (FP64) waves per SIMD: 19.0 / 26.0 KB
    // per 4-wave block). Both take two loads per lane; 96 FP32 points (three) ran 4 % slower, 48
    // FP64 points instead of 32 (fewer chunks for the larger leaves) 4 % faster.
    constexpr int CAP = kFp32 ? kStageBytes / 32 : 48;
    // leaf tests on the matrix cores (leaf_mfma): FP32 sphere counts with one lane per query
    constexpr bool kMfma = kFp32 && KERNEL == OCT_KERNEL_SPHERE && G == 64 && MODE == 0;
    // children judged by their tight boxes; not when the search counters are asked for, which are those of the
    // octree cells, nor for OCT_ALGO_NEIGHBORS, whose box overlaps take few comparisons (5 M tile, r = 1: 1.45
    // against 1.67 ms with boxes)
    constexpr bool kTight = kMfma && !STATS && (ALGO == OCT_ALGO_PRUNE || ALGO == OCT_ALGO_STRUCT);
    constexpr int SMX = S > 16 ? S : 16;                               // largest lane-group count of a leaf
    constexpr int PAD = kUnroll * SMX + SMX;                           // sentinel + row-padding slots after a chunk
    __shared__ uint32_t s_node[kWaves][kStack];
    __shared__ uint64_t s_mask[kWaves][kStack];
    __shared__ uint8_t s_depth[kWaves][kStack];
    __shared__ uint64_t s_leafm[kWaves][8];  // OVERLAP leaf children of the popped node (query masks)
    __shared__ uint8_t s_rmap[kWaves][64];   // remapped leaf: home slot of compacted query r
    __shared__ uint32_t s_rtot[kWaves][64];  // remapped leaf: count of compacted query r
    __shared__ uint64_t s_hits[MODE ? kWaves : 1][MODE ? 64 : 1];     // its hits (lists)
    __shared__ uint64_t s_inm[MODE == 2 ? kWaves : 1][8];             // INSIDE children of the popped node (query masks)
    __shared__ __attribute__((aligned(16))) unsigned char s_stage[kMfma ? 1 : kWaves][kMfma ? 16 : (CAP + PAD) * (kFp32 ? 16 : 32)];
    __shared__ MfmaQueries s_mq[kMfma ? kWaves : 1];

    const uint32_t w = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t g = lane / G, j = lane % G;
    const uint64_t gmask = (G == 64) ? ~0ull : ((1ull << G) - 1ull);
    if (uniform_u32(tile * G) >= a.nq) return;
    const uint32_t slot = tile * G + j;
    // one cloud (root 0), or the wave tile's cloud of a forest and its number of valid slots
    uint32_t cloud = 0, nvt = G, root = 0;
    if (a.tile_info) {
        const uint32_t ti = uniform_u32(a.tile_info[tile]);
        cloud = ti & 0xfffffu, nvt = ti >> 20;
        root = uniform_u32(a.roots[cloud]);
    }
    ConstDouble *radp = const_doubles(a.radtab) + 66 * cloud;  // level radii: radp[3 * level + axis]
    const bool valid = slot < a.nq && j < nvt;
    const uint64_t qbit = 1ull << j;
    float4 *sp32 = reinterpret_cast<float4 *>(&s_stage[kMfma ? 0 : w][0]);
    double4 *sp64 = reinterpret_cast<double4 *>(&s_stage[kMfma ? 0 : w][0]);
    MfmaQueries &mq = s_mq[kMfma ? w : 0];

    Query q;
    uint32_t qid = 0;
    q.x = q.y = q.z = 0.0;
    q.r = 0.0;
    if (valid) {
        qid = a.order ? a.order[slot] : slot;
        if (a.qxyz) {
            q.x = a.qxyz[3 * (size_t)qid], q.y = a.qxyz[3 * (size_t)qid + 1], q.z = a.qxyz[3 * (size_t)qid + 2];
        } else {
            const double4 p = a.p64[a.qidx ? a.qidx[qid] : qid];
            q.x = p.x, q.y = p.y, q.z = p.z;
        }
        q.r = a.qrad ? a.qrad[qid] : a.radius;
    }
    q.R = q.r * q.r;
    q.lox = q.x - q.r, q.loy = q.y - q.r, q.loz = q.z - q.r;
    q.hix = q.x + q.r, q.hiy = q.y + q.r, q.hiz = q.z + q.r;
    if (KERNEL == OCT_KERNEL_CUBE || KERNEL == OCT_KERNEL_SQUARE) box_radii(a, valid, qid, q);
    const float qRf = (float)q.R;

    const float qRs = kTight ? qRf * (a.box_scale * a.box_scale) : 0.0f;
    auto clamp01 = [](float v) -> float { return __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f); };  // an output modifier
    // tight boxes: not for a wave with a query whose scale their margin does not cover
    bool boxes = false;
    if constexpr (kTight) {
        if (a.nbox) {
            ConstNodeBox &B = node_box(a.nbox, 0);
            const float dx = (float)(q.x - B.c[0]), dy = (float)(q.y - B.c[1]), dz = (float)(q.z - B.c[2]);
            const float far = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) + qRf;
            boxes = ballot64(valid && !(q.r >= 0.0 && qRf > a.tight_min && far < 1e29f)) == 0;
        }
    }
    uint32_t cnt = 0, ecnt = 0;
    uint32_t *out = nullptr;  // MODE 2: the next word of the lane's list
    if (MODE == 2 && valid) out = a.entries + a.offsets[qid] * (kRanges ? 2u : 1u);
    uint64_t n_class = 0, n_test = 0, n_recheck = 0, n_cslots = 0, n_tslots = 0;

    // a value of another lane (ds_bpermute)
    auto bperm_u32 = [](uint32_t src_lane, uint32_t v) -> uint32_t {
        return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(src_lane << 2), (int)v);
    };
    auto bperm_f32 = [&](uint32_t src_lane, float v) -> float { return __uint_as_float(bperm_u32(src_lane, __float_as_uint(v))); };
    auto bperm_f64 = [&](uint32_t src_lane, double v) -> double {
        const uint64_t b = (uint64_t)__double_as_longlong(v);
        const uint64_t lo = bperm_u32(src_lane, (uint32_t)b), hi = bperm_u32(src_lane, (uint32_t)(b >> 32));
        return __longlong_as_double((long long)(lo | (hi << 32)));
    };

    auto judge = [&](bool act, const NodeRec &nr, uint32_t d) -> int {
        if (!act) return -1;
        const double rx = radp[3 * d], ry = radp[3 * d + 1], rz = radp[3 * d + 2];
        if (ALGO == OCT_ALGO_NEIGHBORS) return overlap64<KERNEL>(q, nr.cx, nr.cy, nr.cz, rx, ry, rz) ? J_OVERLAP : J_OUTSIDE;
        return classify64<KERNEL>(q, nr.cx, nr.cy, nr.cz, rx, ry, rz);
    };

    // Stage points [base, base + P) of the sorted cloud for 2^lg lane groups: point t goes to group
    // t % 2^lg, row slot t / 2^lg, rows padded with sentinels to iters = a multiple of kUnroll and
    // spaced iters + 1 slots apart when there are several groups (the spare slot turns the rows'
    // 16-byte columns across LDS banks). Group gp then reads slots gp * (iters + (lg > 0)) + k at
    // fixed offsets. All of a chunk's loads are issued before any LDS write (one round trip);
    // loads read a clamped in-range point and the sentinel is selected by value. Returns iters.
    auto stage = [&](uint32_t base, uint32_t P, uint32_t lg) -> uint32_t {
        const uint32_t st = 1u << lg;
        const uint32_t iters = (P + st * kUnroll - 1) / (st * kUnroll) * kUnroll;  // per-lane iterations
        const uint32_t slots = iters * st;
        const uint32_t rs = iters + (lg ? 1u : 0u);
        constexpr int NI = (CAP + kUnroll * SMX + 63) / 64;  // slots <= CAP + kUnroll * SMX - 1
        if (kFp32) {
            // sentinel: t = 1e30 + C (sphere: w = 1e30) or +inf (circle: x = y = 1e30), never
            // inside and above the band
            const float4 sent = KERNEL == OCT_KERNEL_CIRCLE ? make_float4(1e30f, 1e30f, 0.0f, 0.0f)
                                                            : make_float4(0.0f, 0.0f, 0.0f, 1e30f);
            float4 v[NI];
#pragma unroll
            for (int i = 0; i < NI; i++)
                if (64u * i < slots) v[i] = a.p32[base + min(lane + 64u * i, P - 1)];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t t = lane + 64u * i;
                if (64u * i < slots && t < slots) {
                    const bool real = t < P;
                    sp32[(t & (st - 1u)) * rs + (t >> lg)] =
                        make_float4(real ? v[i].x : sent.x, real ? v[i].y : sent.y, real ? v[i].z : sent.z, real ? v[i].w : sent.w);
                }
            }
        } else {
            double4 v[NI];
#pragma unroll
            for (int i = 0; i < NI; i++)
                if (64u * i < slots) v[i] = a.p64[base + min(lane + 64u * i, P - 1)];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t t = lane + 64u * i;
                if (64u * i < slots && t < slots) {
                    const bool real = t < P;
                    sp64[(t & (st - 1u)) * rs + (t >> lg)] =
                        make_double4(real ? v[i].x : __builtin_nan(""), real ? v[i].y : __builtin_nan(""), real ? v[i].z : __builtin_nan(""), 0.0);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        return iters;
    };

    // leaf: the queries in m count the leaf's points. Normally lane group g of each query takes
    // points g, g + S, ... . A leaf wanted by at most half of the wave's queries is remapped: its mc
    // queries are compacted onto groups of Sp = 64 / Gp lanes (Gp = max(4, mc rounded up to a power
    // of 2), so Sp <= 16); lane l serves compacted query r = l % Gp and takes points l / Gp, + Sp, ...;
    // the query's terms are computed in its own lane and fetched with ds_bpermute, and each group's
    // count returns to its query's first lane through LDS. Same tests and band either way.
    auto leaf = [&](uint64_t m, float am, const NodeRec &nr) {
        const uint32_t first = nr.first, last = nr.last;
        if (STATS) n_test += (uint64_t)__popcll(m) * (last - first);
        const uint32_t mc = (uint32_t)__popcll(m);
        const bool rm = a.remap && 2 * mc <= (uint32_t)G;  // wave-uniform
        constexpr uint32_t LS = S == 1 ? 0 : S == 2 ? 1 : S == 4 ? 2 : S == 8 ? 3 : S == 16 ? 4 : S == 32 ? 5 : 6;
        uint32_t lg = 0, lgs = LS, Sp = S, gp = g, src = lane, rank = 0;
        bool ract = (m & qbit) != 0 && valid;
        const bool home = rm && g == 0 && ((m >> j) & 1ull) != 0;
        if (rm) {
            lg = mc <= 4 ? 2u : 32u - (uint32_t)__builtin_clz(mc - 1);
            lgs = 6u - lg;
            Sp = 64u >> lg;
            gp = lane >> lg;
            const uint32_t r = lane & ((1u << lg) - 1u);
            rank = (uint32_t)__popcll(m & (qbit - 1ull));
            if (home) s_rmap[w][rank] = (uint8_t)j;  // slot j's first lane is lane j
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            ract = r < mc;
            src = ract ? (uint32_t)s_rmap[w][r] : lane;
        }
        // a value of the served query: its own lane's, or fetched from the query's lane
        auto qf = [&](float v) -> float { return rm ? bperm_f32(src, v) : v; };
        auto qd = [&](double v) -> double { return rm ? bperm_f64(src, v) : v; };
        auto fetch_query = [&]() {
            Query qr = q;
            if (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE) {
                qr.x = qd(q.x), qr.y = qd(q.y), qr.R = qd(q.R);
                if (KERNEL == OCT_KERNEL_SPHERE) qr.z = qd(q.z);
            } else {
                qr.lox = qd(q.lox), qr.hix = qd(q.hix), qr.loy = qd(q.loy), qr.hiy = qd(q.hiy);
                if (KERNEL == OCT_KERNEL_CUBE) qr.loz = qd(q.loz), qr.hiz = qd(q.hiz);
            }
            return qr;
        };
        uint32_t lc = 0;
        if (kFp32) {
            // t = fma(ax, -2bx, fma(ay, -2by, fma(az, -2bz, w + C))) (circle: fma(ax, ax - 2bx,
            // fma(ay, ay - 2by, C))) with C = fl32(fl32(hw - fl32(R)) + fl32(|b|^2)) approximates
            // u + hw, u = |p - q|^2 - R. Only b = fl32(q - c) is formed in FP64; the rest of the set-up
            // is FP32. Bounding the error for any association of the five terms, with every product
            // and sum rounded to nearest or toward zero (u' = 2^-23), and with the representation
            // errors of a, b, w and the FP32 set-up (unit u = 2^-24):
            //   |t - (u + hw)| <= u (25 amax + 28 |b|^2 + 13 R + 12 hw) < 32 u (amax + |b|^2 + R);
            // the circle form's fl32(ax - 2bx) adds at most u (2 amax + |b|^2). hw = 2^-18 fl32(fl32(amax +
            // fl32|b|^2) + fl32 R) >= 2 * 32 u (amax + |b|^2 + R)(1 - 5u) covers both with a factor-2
            // margin. Hence t <= 0 (sign bit set, -0 included) is inside, t > 2 hw is outside, and
            // 0 <= t <= 2 hw - an unsigned compare of the bit patterns, which also sends +0 there - is
            // re-tested in FP64. Slots past the leaf are sentinels (t ~ 1e30 or +inf, above 2 hw). A
            // leaf/query pair with amax + |b|^2 + R >= 1e30 (or not finite: a non-finite point makes
            // amax = inf) or <= 1e-30 is re-tested in FP64 outright (lim = ~0), so no term can overflow and
            // what denormal products lose stays below the band.
            const float bx = (float)(q.x - nr.cx), by = (float)(q.y - nr.cy), bz = (float)(q.z - nr.cz);
            const float b2 = KERNEL == OCT_KERNEL_SPHERE ? __builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz))
                                                         : __builtin_fmaf(bx, bx, by * by);
            const float sum = (am + b2) + qRf;
            const float hw = 3.814697265625e-06f * sum;  // 2^-18
            const float C = qf((hw - qRf) + b2);
            const uint32_t lim = __float_as_uint(qf(__uint_as_float(fp32_range(sum) ? __float_as_uint(2.0f * hw) : 0xffffffffu)));
            const float ux = qf(-2.0f * bx), uy = qf(-2.0f * by);
            const float uz = KERNEL == OCT_KERNEL_SPHERE ? qf(-2.0f * bz) : 0.0f;
            uint32_t c8 = 0, c8b = 0, mnb = 0xffffffffu;
            for (uint32_t base = first; base < last; base += CAP) {
                const uint32_t P = (last - base) < (uint32_t)CAP ? (last - base) : (uint32_t)CAP;
                const uint32_t iters = stage(base, P, lgs);
                const float4 *pl = sp32 + gp * (iters + (lgs ? 1u : 0u));
                for (uint32_t k = 0; k < iters; k += kUnroll, pl += kUnroll) {
                    const float4 p0 = pl[0], p1 = pl[1], p2 = pl[2], p3 = pl[3];
                    float t0, t1, t2, t3;
                    if (KERNEL == OCT_KERNEL_SPHERE) {
                        t0 = __builtin_fmaf(p0.x, ux, __builtin_fmaf(p0.y, uy, __builtin_fmaf(p0.z, uz, p0.w + C)));
                        t1 = __builtin_fmaf(p1.x, ux, __builtin_fmaf(p1.y, uy, __builtin_fmaf(p1.z, uz, p1.w + C)));
                        t2 = __builtin_fmaf(p2.x, ux, __builtin_fmaf(p2.y, uy, __builtin_fmaf(p2.z, uz, p2.w + C)));
                        t3 = __builtin_fmaf(p3.x, ux, __builtin_fmaf(p3.y, uy, __builtin_fmaf(p3.z, uz, p3.w + C)));
                    } else {
                        t0 = __builtin_fmaf(p0.x, p0.x + ux, __builtin_fmaf(p0.y, p0.y + uy, C));
                        t1 = __builtin_fmaf(p1.x, p1.x + ux, __builtin_fmaf(p1.y, p1.y + uy, C));
                        t2 = __builtin_fmaf(p2.x, p2.x + ux, __builtin_fmaf(p2.y, p2.y + uy, C));
                        t3 = __builtin_fmaf(p3.x, p3.x + ux, __builtin_fmaf(p3.y, p3.y + uy, C));
                    }
                    const uint32_t d0 = __float_as_uint(t0), d1 = __float_as_uint(t1);
                    const uint32_t d2 = __float_as_uint(t2), d3 = __float_as_uint(t3);
                    // two accumulators: each v_bcnt adds into its own (one add3 fewer per 4 tests)
                    c8 = __builtin_popcount(__builtin_amdgcn_perm(d0, d1, 0x0c0c0b09u)) + c8;
                    c8b = __builtin_popcount(__builtin_amdgcn_perm(d2, d3, 0x0c0c0b09u)) + c8b;
                    mnb = min(min(mnb, d0), d1);
                    mnb = min(min(mnb, d2), d3);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            lc = (c8 + c8b) >> 3;
            const bool band = ract && mnb <= lim;
            if (ballot64(band)) {  // rare: exact FP64 re-count of this lane's share of the leaf
                const Query qr = fetch_query();
                if (band) {
                    lc = 0;
                    for (uint32_t i = first + gp; i < last; i += Sp) {
                        const double4 pd = a.p64[i];
                        lc += inside64<KERNEL>(qr, pd.x, pd.y, pd.z);
                        if (STATS) n_recheck++;
                    }
                }
            }
        } else {
            const Query qr = fetch_query();
            for (uint32_t base = first; base < last; base += CAP) {
                const uint32_t P = (last - base) < (uint32_t)CAP ? (last - base) : (uint32_t)CAP;
                const uint32_t iters = stage(base, P, lgs);
                const double4 *pl = sp64 + gp * (iters + (lgs ? 1u : 0u));
                uint32_t c0 = 0, c1 = 0, c2 = 0, c3 = 0;
                for (uint32_t k = 0; k < iters; k += kUnroll, pl += kUnroll) {
                    const double4 p0 = pl[0], p1 = pl[1], p2 = pl[2], p3 = pl[3];
                    c0 += inside64<KERNEL>(qr, p0.x, p0.y, p0.z) ? 1u : 0u;
                    c1 += inside64<KERNEL>(qr, p1.x, p1.y, p1.z) ? 1u : 0u;
                    c2 += inside64<KERNEL>(qr, p2.x, p2.y, p2.z) ? 1u : 0u;
                    c3 += inside64<KERNEL>(qr, p3.x, p3.y, p3.z) ? 1u : 0u;
                }
                lc += (c0 + c1) + (c2 + c3);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (!ract) lc = 0;
        if (rm) {
            // butterfly over the lanes that served one compacted query (lane % 2^lg equal, lg >= 2)
            if (lg <= 2) lc += lane_xor<4>(lc);
            if (lg <= 3) lc += lane_xor<8>(lc);
            if (lg <= 4) lc += lane_xor<16>(lc);
            lc += lane_xor32(lc);
            if (ract && gp == 0) s_rtot[w][lane] = lc;  // lane = r for the group's first lane
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            lc = home ? s_rtot[w][rank] : 0u;
        }
        cnt += lc;
        if (STATS) n_tslots += 64ull * ((last - first + Sp - 1) / Sp);
    };

    // Tight boxes (kTight): a child whose points' box lies inside a query's sphere, or outside it, by a margin of
    // 2^-18 (ext2 + |b|^2 + R) needs no further look, whatever the octree cells say: every point then passes, or
    // fails, its own test, and no cell that holds it can have been judged otherwise up to rounding. The margin
    // is 64 u (u = 2^-24) of that sum; the FP32 distances to the box are within 45 u. Between, a child is
    // descended into or its points are tested. The FP64 judgement of the cells (the reference's answer) can
    // differ from the points' own tests only where a point lies on the sphere to the last FP64 bits: such a point
    // is in the band of its leaf's test, and its lane's points are then decided by path_class, the reference's
    // walk itself. This holds for points inside their cells; a node with others below it has no boxes (ext2 is
    // infinite) and is judged by its cells. tie_scale sqrt(S) + 2^-46 S bounds the cells' and points' rounding (S as above, coordinates
    // up to 2^46 tie_scale), and S > tight_min keeps it below the margin's slack.
    //
    // 50 M tile, r = 2.5 (all points): 1418 point tests per query instead of 1684, 38.2 -> 29.9 ms with leaf_mfma;
    // leaf_mfma alone, the cells judged in FP64, 36.8 ms.

    // How the reference's walk from the root decides the leaf that starts at point `first` for query qr:
    // INSIDE or OUTSIDE at a node on the way, or OVERLAP down to the leaf. The whole wave calls it.
    auto path_class = [&](const Query &qr, uint32_t first) -> int {
        int cls = J_OVERLAP;
        uint32_t node = root;
        for (uint32_t d = 0; d <= kMaxDepth; d++) {
            const NodeRec nr = a.nodes[node];
            if (cls == J_OVERLAP) {
                const double rx = radp[3 * d], ry = radp[3 * d + 1], rz = radp[3 * d + 2];
                if (ALGO == OCT_ALGO_NEIGHBORS)
                    cls = overlap64<KERNEL>(qr, nr.cx, nr.cy, nr.cz, rx, ry, rz) ? J_OVERLAP : J_OUTSIDE;
                else
                    cls = classify64<KERNEL>(qr, nr.cx, nr.cy, nr.cz, rx, ry, rz);
            }
            const uint32_t c0 = uniform_u32(a.child[node]);
            if (c0 == 0) break;
            const NodeRec cr = a.nodes[c0 + (lane & 7u)];
            const uint64_t at = ballot64(cr.first <= first && first < cr.last) & 0xffull;
            if (!at) break;
            node = c0 + (uint32_t)__builtin_ctzll(at);
        }
        return cls;
    };

    // The leaf tests on the matrix cores. t of leaf() is the product of a point's (x, y, z, w) with a query's
    // (-2 b, 1) plus its C: v_mfma_f32_16x16x4 makes it for 16 points and 16 queries. The queries that want the
    // leaf (m) are compacted into columns, their terms go through LDS once; a leaf's 64 points are one load,
    // turned into four row operands by lane swaps. Lane 16 g + c of a result holds points 4 g .. 4 g + 3 and
    // query c; hits and the band are counted per lane as in leaf(), whose error bound holds for any order of the
    // sum and either rounding. Vector FMAs run at the matrix rate (2 cycles per wave here), so the gain is
    // what surrounds them: 4 LDS reads and a staging pass fewer per 4 tests. Here 2-operand FP32 and integer
    // instructions on VGPRs take 2.5 cycles, all others (3 operands, scalar operands, compares, min, FP64) 4.3.
    // tight: the leaf was reached through its parent's tight boxes, whose conditions (a finite am below 1e30 in a box
    // below 1e15, a query nearer than 3.2e14 to its centre, R above 1e-30) keep every term within FP32. Leaves
    // reached by their cells can hold points beyond FP32 and NaNs, whatever the wave's queries. Their ties need no
    // walk: a node has boxes where all below it have them, so a leaf without them had every ancestor's cell judged.
    auto leaf_mfma = [&](const uint64_t m, const float am, const NodeRec &nr, const bool tight) {
        const uint32_t first = nr.first, last = nr.last;
        if (STATS) n_test += (uint64_t)__popcll(m) * (last - first);
        const uint32_t mc = (uint32_t)__popcll(m);
        const bool act = __builtin_amdgcn_inverse_ballot_w64(m);
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const float4 sent = make_float4(0.0f, 0.0f, 0.0f, 1e30f);  // outside every query, above the band
        float4 v = sent;
        if (lane < last - first) v = (a.p32 + first)[lane];
        if (act) {
            const float bx = (float)(q.x - nr.cx), by = (float)(q.y - nr.cy), bz = (float)(q.z - nr.cz);
            const float b2 = __builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz));
            const float sum = (am + b2) + qRf;
            const float hw = 3.814697265625e-06f * sum;  // 2^-18
            const float C = (hw - qRf) + b2;
            float lim = 2.0f * hw;
            if (!tight && !fp32_range(sum)) lim = __uint_as_float(0xffffffffu);
            mq.u[rank] = make_float4(-2.0f * bx, -2.0f * by, -2.0f * bz, 1.0f);
            mq.c[rank] = make_float4(C, C, C, C);
            mq.lh[rank] = make_uint2(__float_as_uint(lim), lane);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t nt = (mc + 15) >> 4, col = lane & 15;
        for (uint32_t base = first; base < last; base += 64) {
            const uint32_t P = (last - base) < 64u ? (last - base) : 64u;
            if (base != first) {
                v = sent;
                if (lane < P) v = (a.p32 + base)[lane];
            }
            // the four terms of points 16 i .. 16 i + 15 into one register
            const u32x2 s02 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.x), __float_as_uint(v.z), false, false);
            const u32x2 s13 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.y), __float_as_uint(v.w), false, false);
            const u32x2 a01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
            const u32x2 a23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
            const float A[4] = {__uint_as_float(a01[0]), __uint_as_float(a01[1]), __uint_as_float(a23[0]), __uint_as_float(a23[1])};
            uint32_t band = 0;  // bit t: a point of this lane's is in the band of its query of tile t
            uint32_t acc = 0;   // byte t: 8 x the hits of this lane's points and its query of tile t (at most 16)
            auto rows = [&](auto rt_c) {
                constexpr int RT = decltype(rt_c)::value;
                const float *pu = reinterpret_cast<const float *>(mq.u) + col * 4 + (lane >> 4);
                const float4 *pc = mq.c + col;
                for (uint32_t t = 0; t < nt; t++, pu += 64, pc += 16) {
                    const float B = *pu;
                    const float4 c4 = *pc;
                    const uint32_t lim = reinterpret_cast<const MfmaQueries::Lim *>(pc + 64)->lim;  // mq.lh
                    const f32x4 cq = {c4.x, c4.y, c4.z, c4.w};
                    f32x4 d[RT];
#pragma unroll
                    for (int i = 0; i < RT; i++) d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[i], B, cq, 0, 0, 0);
                    uint32_t c8 = 0, mnb = 0xffffffffu;
#pragma unroll
                    for (int i = 0; i < RT; i++) {
                        const uint32_t d0 = __float_as_uint(d[i][0]), d1 = __float_as_uint(d[i][1]);
                        const uint32_t d2 = __float_as_uint(d[i][2]), d3 = __float_as_uint(d[i][3]);
                        c8 = __builtin_popcount(__builtin_amdgcn_perm(d0, d1, 0x0c0c0b09u)) + c8;
                        c8 = __builtin_popcount(__builtin_amdgcn_perm(d2, d3, 0x0c0c0b09u)) + c8;
                        mnb = min(min(mnb, d0), d1);
                        mnb = min(min(mnb, d2), d3);
                    }
                    const uint64_t bm = ballot64(mnb <= lim);
                    if (bm) band |= __builtin_amdgcn_inverse_ballot_w64(bm) ? 1u << t : 0u;
                    acc += c8 << (8 * t);
                }
                if (STATS) n_tslots += 256ull * RT * nt;
            };
            if (P > 48)
                rows(std::integral_constant<int, 4>{});
            else if (P > 32)
                rows(std::integral_constant<int, 3>{});
            else if (P > 16)
                rows(std::integral_constant<int, 2>{});
            else
                rows(std::integral_constant<int, 1>{});
            for (uint32_t t = 0; ballot64(band >> t); t++) {  // rare: exact FP64 counts of a lane's points
                const bool redo = ((band >> t) & 1u) && col + 16 * t < mc;
                if (!ballot64(redo)) continue;
                const uint32_t src = mq.lh[col + 16 * t].home & 63u;
                Query qr = q;
                qr.x = bperm_f64(src, q.x), qr.y = bperm_f64(src, q.y), qr.z = bperm_f64(src, q.z);
                qr.r = bperm_f64(src, q.r), qr.R = qr.r * qr.r;
                bool tie = false;
                uint32_t np = 0, c8 = 0;
                if (redo) {
                    const double bx = qr.x - nr.cx, by = qr.y - nr.cy, bz = qr.z - nr.cz;
                    const double sc = ((double)am + (bx * bx + by * by + bz * bz)) + qr.R;
                    const double thr = a.tie_scale * (double)sqrtf((float)sc) + 1.4210854715202004e-14 * sc;  // 2^-46
                    for (uint32_t i = 4 * (lane >> 4); i < P; i = (i & 3u) == 3u ? i + 13u : i + 1u, np++) {
                        const double4 pd = a.p64[base + i];
                        c8 += inside64<KERNEL>(qr, pd.x, pd.y, pd.z) ? 8u : 0u;
                        const double dx = pd.x - qr.x, dy = pd.y - qr.y, dz = pd.z - qr.z;
                        tie |= !(fabs(((dx * dx + dy * dy) + dz * dz) - qr.R) > thr);
                        if (STATS) n_recheck++;
                    }
                }
                if (tight && ballot64(tie)) {
                    qr.lox = qr.x - qr.r, qr.loy = qr.y - qr.r, qr.loz = qr.z - qr.r;
                    qr.hix = qr.x + qr.r, qr.hiy = qr.y + qr.r, qr.hiz = qr.z + qr.r;
                    const int cls = path_class(qr, first);
                    if (tie && cls != J_OVERLAP) c8 = cls == J_INSIDE ? 8u * np : 0u;
                }
                if (redo) acc = (acc & ~(0xffu << (8 * t))) | (c8 << (8 * t));
            }
            // word (column, row group) of the hits: a query's four words hold its count in byte rank / 16
            mq.acc[4 * col + (lane >> 4)] = acc >> 3;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (act) {
                const uint4 h = *reinterpret_cast<const uint4 *>(mq.acc + 4 * (rank & 15u));
                cnt += ((h.x + h.y + h.z + h.w) >> (8 * (rank >> 4))) & 0xffu;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };

    // Lists: a leaf's points are tested as for counts, but each lane collects its hits as a bit mask, 64 points
    // (48 in FP64) at a time: one shift per test instead of a popcount per four. A remapped leaf's lanes take
    // contiguous points (a power of two per lane), so their masks are shifted into place and OR-ed over the
    // lanes of a query. Counts and runs are then popcounts, and a list's words are the set bits of the mask
    // (indices), or of the mask XOR its neighbour (a run's first point and the one after its last).
    auto leaf_lists = [&](uint64_t m, float am, const NodeRec &nr) {
        const uint32_t first = nr.first, last = nr.last;
        if (STATS) n_test += (uint64_t)__popcll(m) * (last - first);
        const uint32_t mc = (uint32_t)__popcll(m);
        const bool rm = a.remap && 2 * mc <= 64;  // wave-uniform
        const bool act = ((m >> lane) & 1ull) != 0 && valid;  // this lane's query wants the leaf
        uint32_t lg = 0, lgs = 0, gp = 0, src = lane, rank = 0;
        bool ract = act;
        if (rm) {
            lg = mc <= 4 ? 2u : 32u - (uint32_t)__builtin_clz(mc - 1);
            lgs = 6u - lg;
            gp = lane >> lg;
            const uint32_t r = lane & ((1u << lg) - 1u);
            rank = (uint32_t)__popcll(m & (qbit - 1ull));
            if (act) s_rmap[w][rank] = (uint8_t)lane;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            ract = r < mc;
            src = ract ? (uint32_t)s_rmap[w][r] : lane;
        }
        auto qf = [&](float v) -> float { return rm ? bperm_f32(src, v) : v; };
        auto qd = [&](double v) -> double { return rm ? bperm_f64(src, v) : v; };
        auto fetch_query = [&]() {
            Query qr = q;
            if (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CIRCLE) {
                qr.x = qd(q.x), qr.y = qd(q.y), qr.R = qd(q.R);
                if (KERNEL == OCT_KERNEL_SPHERE) qr.z = qd(q.z);
            } else {
                qr.lox = qd(q.lox), qr.hix = qd(q.hix), qr.loy = qd(q.loy), qr.hiy = qd(q.hiy);
                if (KERNEL == OCT_KERNEL_CUBE) qr.loz = qd(q.loz), qr.hiz = qd(q.hiz);
            }
            return qr;
        };
        float C = 0.f, ux = 0.f, uy = 0.f, uz = 0.f;
        uint32_t lim = 0;
        Query qr = q;
        if (kFp32) {  // the count leaf's terms and bound
            const float bx = (float)(q.x - nr.cx), by = (float)(q.y - nr.cy), bz = (float)(q.z - nr.cz);
            const float b2 = KERNEL == OCT_KERNEL_SPHERE ? __builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz))
                                                         : __builtin_fmaf(bx, bx, by * by);
            const float sum = (am + b2) + qRf;
            const float hw = 3.814697265625e-06f * sum;  // 2^-18
            C = qf((hw - qRf) + b2);
            lim = __float_as_uint(qf(__uint_as_float(fp32_range(sum) ? __float_as_uint(2.0f * hw) : 0xffffffffu)));
            ux = qf(-2.0f * bx), uy = qf(-2.0f * by);
            uz = KERNEL == OCT_KERNEL_SPHERE ? qf(-2.0f * bz) : 0.0f;
        } else {
            qr = fetch_query();
        }
        bool open = false;  // range lists: the lane's current run reaches the chunk's first point
        for (uint32_t base = first; base < last; base += CAP) {
            const uint32_t P = (last - base) < (uint32_t)CAP ? (last - base) : (uint32_t)CAP;
            const uint32_t per = (P + (1u << lgs) - 1) >> lgs;  // points per lane, then a multiple of 4 or a power of two
            const uint32_t iters = lgs == 0 ? (P + 3u) & ~3u : (per <= 4 ? 4u : per <= 8 ? 8u : per <= 16 ? 16u : 32u);
            const uint32_t li = 31u - (uint32_t)__builtin_clz(iters);  // lgs > 0: log2(iters)
            const uint32_t rs = lgs ? iters + 1 : 0u;                  // rows of lane groups, one slot apart in the banks
            const uint32_t slots = iters << lgs;
            constexpr int NI = 1;
            {
                const uint32_t t = lane;
                const bool real = t < P;
                const uint32_t at = lgs ? (t >> li) * rs + (t & (iters - 1)) : t;
                if (kFp32) {
                    const float4 v = a.p32[base + min(t, P - 1)];
                    if (t < slots)
                        sp32[at] = real ? v
                                        : (KERNEL == OCT_KERNEL_CIRCLE ? make_float4(1e30f, 1e30f, 0.0f, 0.0f)
                                                                       : make_float4(0.0f, 0.0f, 0.0f, 1e30f));
                } else {
                    const double4 v = a.p64[base + min(t, P - 1)];
                    if (t < slots) sp64[at] = make_double4(real ? v.x : __builtin_nan(""), real ? v.y : __builtin_nan(""), real ? v.z : __builtin_nan(""), 0.0);
                }
            }
            static_assert(NI == 1 && CAP <= 64, "one load per lane and chunk");
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            uint32_t mnb = 0xffffffffu;
            // hits of points [k0, k1) of the lane's row, first point in the highest of the k1 - k0 low bits
            auto hits = [&](const uint32_t k0, const uint32_t k1) -> uint32_t {
                uint32_t hm = 0;
                if (kFp32) {
                    const float4 *pl = sp32 + gp * rs + k0;
                    for (uint32_t k = k0; k < k1; k += 4, pl += 4) {
                        const float4 p0 = pl[0], p1 = pl[1], p2 = pl[2], p3 = pl[3];
                        float t0, t1, t2, t3;
                        if (KERNEL == OCT_KERNEL_SPHERE) {
                            t0 = __builtin_fmaf(p0.x, ux, __builtin_fmaf(p0.y, uy, __builtin_fmaf(p0.z, uz, p0.w + C)));
                            t1 = __builtin_fmaf(p1.x, ux, __builtin_fmaf(p1.y, uy, __builtin_fmaf(p1.z, uz, p1.w + C)));
                            t2 = __builtin_fmaf(p2.x, ux, __builtin_fmaf(p2.y, uy, __builtin_fmaf(p2.z, uz, p2.w + C)));
                            t3 = __builtin_fmaf(p3.x, ux, __builtin_fmaf(p3.y, uy, __builtin_fmaf(p3.z, uz, p3.w + C)));
                        } else {
                            t0 = __builtin_fmaf(p0.x, p0.x + ux, __builtin_fmaf(p0.y, p0.y + uy, C));
                            t1 = __builtin_fmaf(p1.x, p1.x + ux, __builtin_fmaf(p1.y, p1.y + uy, C));
                            t2 = __builtin_fmaf(p2.x, p2.x + ux, __builtin_fmaf(p2.y, p2.y + uy, C));
                            t3 = __builtin_fmaf(p3.x, p3.x + ux, __builtin_fmaf(p3.y, p3.y + uy, C));
                        }
                        const uint32_t d0 = __float_as_uint(t0), d1 = __float_as_uint(t1);
                        const uint32_t d2 = __float_as_uint(t2), d3 = __float_as_uint(t3);
                        hm = __builtin_amdgcn_alignbit(hm, d0, 31);  // hm << 1 | sign
                        hm = __builtin_amdgcn_alignbit(hm, d1, 31);
                        hm = __builtin_amdgcn_alignbit(hm, d2, 31);
                        hm = __builtin_amdgcn_alignbit(hm, d3, 31);
                        mnb = min(min(mnb, d0), d1);
                        mnb = min(min(mnb, d2), d3);
                    }
                } else {
                    const double4 *pl = sp64 + gp * rs + k0;
                    for (uint32_t k = k0; k < k1; k += 4, pl += 4) {
                        const double4 p0 = pl[0], p1 = pl[1], p2 = pl[2], p3 = pl[3];
                        hm = hm + hm + (inside64<KERNEL>(qr, p0.x, p0.y, p0.z) ? 1u : 0u);
                        hm = hm + hm + (inside64<KERNEL>(qr, p1.x, p1.y, p1.z) ? 1u : 0u);
                        hm = hm + hm + (inside64<KERNEL>(qr, p2.x, p2.y, p2.z) ? 1u : 0u);
                        hm = hm + hm + (inside64<KERNEL>(qr, p3.x, p3.y, p3.z) ? 1u : 0u);
                    }
                }
                return __builtin_bitreverse32(hm) >> ((32u - (k1 - k0)) & 31u);
            };
            const uint32_t n0 = iters < 32u ? iters : 32u;
            uint64_t hm = hits(0, n0);
            if (iters > 32u) hm |= (uint64_t)hits(32, iters) << 32;
            if (STATS) n_tslots += 64ull * iters;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (kFp32) {
                const bool band = ract && mnb <= lim;
                if (ballot64(band)) {  // rare: exact FP64 decisions for this lane's share of the chunk
                    const Query qe = fetch_query();
                    if (band) {
                        hm = 0;
                        for (uint32_t k = 0; k < iters && gp * iters + k < P; k++) {
                            const double4 pd = a.p64[base + gp * iters + k];
                            hm |= (uint64_t)(inside64<KERNEL>(qe, pd.x, pd.y, pd.z) ? 1u : 0u) << k;
                            if (STATS) n_recheck++;
                        }
                    }
                }
            }
            if (!ract) hm = 0;
            if (rm) {
                hm <<= gp * iters;
                uint32_t hl = (uint32_t)hm, hh = (uint32_t)(hm >> 32);
                if (lg <= 2) hl |= lane_xor<4>(hl), hh |= lane_xor<4>(hh);
                if (lg <= 3) hl |= lane_xor<8>(hl), hh |= lane_xor<8>(hh);
                if (lg <= 4) hl |= lane_xor<16>(hl), hh |= lane_xor<16>(hh);
                hl |= lane_xor32(hl), hh |= lane_xor32(hh);
                if (ract && gp == 0) s_hits[w][lane] = ((uint64_t)hh << 32) | hl;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                hm = act ? s_hits[w][rank] : 0ull;
            }
            const uint64_t pm = P == 64 ? ~0ull : (1ull << P) - 1ull;
            hm &= pm;
            const uint64_t pr = (hm << 1) | (open ? 1ull : 0ull);
            if (MODE == 1) {
                cnt += (uint32_t)__popcll(hm);
                ecnt += (uint32_t)__popcll(hm & ~pr);
            } else {
                const uint64_t words = kRanges ? (hm ^ pr) & pm : hm;
                uint32_t wl = (uint32_t)words, wh = (uint32_t)(words >> 32);
                while (wl) {
                    *out++ = base + (uint32_t)__builtin_ctz(wl);
                    wl &= wl - 1u;
                }
                while (wh) {
                    *out++ = base + 32u + (uint32_t)__builtin_ctz(wh);
                    wh &= wh - 1u;
                }
            }
            if (kRanges) open = ((hm >> (P - 1u)) & 1ull) != 0;
        }
        if (MODE == 2 && kRanges && open) *out++ = last;  // a run ends with its leaf
    };

    // The 8 children of a popped node are judged from per-axis terms: they take two centre values
    // per axis (NodeExt), so |q - c|, the kernel-box bounds and the squared extents are computed
    // once per axis value and combined per child, in the reference's operation order, e.g. for the
    // sphere (ex*ex + ey*ey) + ez*ez with ex = |q.x - cx| + rx (kernel_3d.hpp:181-223). Each lane
    // judges all 8 children for its own query (the S lanes of a query agree). Every comparison
    // becomes a lane mask at once (ballot), so the per-child decisions are scalar-unit operations
    // on masks, and the results are lane masks: inm[c] (INSIDE) and ovm[c] (OVERLAP), both within
    // actm, the lanes whose query wants the popped node.
    auto judge8 = [&](ConstNodeExt &E, uint32_t d, uint64_t actm, uint64_t (&inm)[8], uint64_t (&ovm)[8]) {
        if (ALGO == OCT_ALGO_APPROX && d > a.approx_level) {
            // neighborsApprox beyond its precision level: every child whole, or none
            // (linear_octree.hpp:987-994)
#pragma unroll
            for (int c = 0; c < 8; c++) inm[c] = a.approx_upper ? actm : 0ull, ovm[c] = 0ull;
            return;
        }
        const double rx = radp[3 * d], ry = radp[3 * d + 1], rz = radp[3 * d + 2];
        constexpr bool is3d = (KERNEL == OCT_KERNEL_SPHERE || KERNEL == OCT_KERNEL_CUBE);
        if (ALGO == OCT_ALGO_NEIGHBORS || KERNEL == OCT_KERNEL_CUBE || KERNEL == OCT_KERNEL_SQUARE) {
            // boxOverlap (kernel_3d.hpp:100-115, kernel_2d.hpp:29-41) and the box kernels'
            // boxIntersect (kernel_3d.hpp:277-302, kernel_2d.hpp:195-218): per-axis comparisons
            uint64_t ox[2], oy[2], oz[2], ix[2], iy[2], iz[2];
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const double hx = E.ax[b] + rx, lx = E.ax[b] - rx, hy = E.ax[2 + b] + ry, ly = E.ax[2 + b] - ry;
                const double hz = E.ax[4 + b] + rz, lz = E.ax[4 + b] - rz;
                ox[b] = ballot64(hx < q.lox || lx > q.hix);
                oy[b] = ballot64(hy < q.loy || ly > q.hiy);
                oz[b] = is3d ? ballot64(hz < q.loz || lz > q.hiz) : 0ull;
                ix[b] = ballot64(hx <= q.hix && lx >= q.lox);
                iy[b] = ballot64(hy <= q.hiy && ly >= q.loy);
                iz[b] = is3d ? ballot64(hz <= q.hiz && lz >= q.loz) : ~0ull;
            }
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int bx = c & 1, by = (c >> 1) & 1, bz = (c >> 2) & 1;
                const uint64_t keep = actm & ~(ox[bx] | oy[by] | oz[bz]);
                const uint64_t inside = ALGO != OCT_ALGO_NEIGHBORS ? keep & ix[bx] & iy[by] & iz[bz] : 0ull;
                inm[c] = inside;
                ovm[c] = keep & ~inside;
            }
        } else {
            // sphere / circle boxIntersect (kernel_3d.hpp:181-223, kernel_2d.hpp:107-144)
            double e2x[2], e2y[2], e2z[2], m2x[2], m2y[2], m2z[2];
            uint64_t ox[2], oy[2], oz[2], nx[2], ny[2], nz[2];
            const double mdx = q.r + rx, mdy = q.r + ry, mdz = q.r + rz;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const double dx = fabs(q.x - E.ax[b]), dy = fabs(q.y - E.ax[2 + b]);
                ox[b] = ballot64(dx > mdx), oy[b] = ballot64(dy > mdy);
                nx[b] = ballot64(dx < rx), ny[b] = ballot64(dy < ry);
                const double ex = dx + rx, ey = dy + ry;
                e2x[b] = ex * ex, e2y[b] = ey * ey;
                const double fx = dmax0(dx - rx), fy = dmax0(dy - ry);
                m2x[b] = fx * fx, m2y[b] = fy * fy;
                if (is3d) {
                    const double dz = fabs(q.z - E.ax[4 + b]);
                    oz[b] = ballot64(dz > mdz), nz[b] = ballot64(dz < rz);
                    const double ez = dz + rz, fz = dmax0(dz - rz);
                    e2z[b] = ez * ez, m2z[b] = fz * fz;
                } else {
                    oz[b] = nz[b] = 0ull, e2z[b] = m2z[b] = 0.0;
                }
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {  // (bx, by) pairs; each partial sum serves both z halves
                const int bx = k & 1, by = k >> 1;
                const double sxy = e2x[bx] + e2y[by], txy = m2x[bx] + m2y[by];
                const uint64_t oxy = ox[bx] | oy[by], nxy = nx[bx] & ny[by], nxoy = nx[bx] | ny[by];
#pragma unroll
                for (int bz = 0; bz < (is3d ? 2 : 1); bz++) {
                    const int c = k | (bz << 2);
                    const uint64_t keep = actm & ~(oxy | oz[bz]);
                    const double smax = is3d ? sxy + e2z[bz] : sxy;
                    const double smin = is3d ? txy + m2z[bz] : txy;
                    const uint64_t inside = keep & ballot64(smax <= q.R);
                    // two of the three axes inside the node's slab: (nx && ny) || (nz && (nx || ny))
                    const uint64_t two = is3d ? (nxy | (nz[bz] & nxoy)) : nxy;
                    inm[c] = inside;
                    ovm[c] = keep & ~inside & (two | ballot64(smin <= q.R));
                    if (!is3d) {  // 2-D kernels: the z half of the children repeats the judgement
                        inm[c | 4] = inm[c];
                        ovm[c | 4] = ovm[c];
                    }
                }
            }
        }
    };

    // root (singleTraversal, linear_octree.hpp:655-662); group 0 owns the root's INSIDE count.
    // Stack entries hold the FIRST CHILD of an OVERLAP internal node; its NodeExt record is one
    // uniform load.
    uint32_t sp = 0;
    uint32_t overflow = 0;  // wave-uniform: a push found the stack full (cannot happen within 21 levels)
    {
        const NodeRec nr = a.nodes[root];
        const int jr = judge(valid, nr, 0);
        if (STATS) n_class += __popcll(ballot64(valid) & gmask), n_cslots += 64;
        if (g == 0 && jr == J_INSIDE) {
            cnt += nr.last - nr.first, ecnt++;
            if (MODE == 2) {
                if (kRanges)
                    *out++ = nr.first, *out++ = nr.last;
                else
                    for (uint32_t i = nr.first; i < nr.last; i++) *out++ = i;
            }
        }
        const uint64_t ov = ballot64(jr == J_OVERLAP) & gmask;
        if (ov) {
            const uint32_t c0 = uniform_u32(a.child[root]);
            if (c0 == 0) {
                NodeRec ur;
                ur.cx = nr.cx, ur.cy = nr.cy, ur.cz = nr.cz;
                ur.first = uniform_u32(nr.first), ur.last = uniform_u32(nr.last);
                if (ur.last > ur.first) {
                    if constexpr (kMfma)
                        leaf_mfma(ov, a.amax[root], ur, false);
                    else if constexpr (MODE == 0)
                        leaf(ov, a.amax[root], ur);
                    else
                        leaf_lists(ov, a.amax[root], ur);
                }
            } else {
                s_node[w][0] = c0, s_mask[w][0] = ov, s_depth[w][0] = 0;
                sp = 1;
            }
        }
    }
    while (sp > 0) {
        sp--;
        const uint32_t fc = uniform_u32(s_node[w][sp]);
        const uint64_t m = uniform_u64(s_mask[w][sp]);
        const uint32_t d = uniform_u32(s_depth[w][sp]) + 1;  // the children's level
        ConstNodeExt &E = node_ext(a.next, (fc - 1) >> 3);
        // lanes whose query wants the node: bit j of m for lane g * G + j
        const uint64_t actm = G == 64 ? m : ballot64((m & qbit) != 0);
        if constexpr (kTight) {
            ConstNodeBox &B = node_box(a.nbox, (fc - 1) >> 3);
            if (boxes && B.ext2 < 1e29f) {
                const float bx = a.box_scale * (float)(q.x - B.c[0]), by = a.box_scale * (float)(q.y - B.c[1]);
                const float bz = a.box_scale * (float)(q.z - B.c[2]);
                const float b2 = __builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz));
                const float hw = 3.814697265625e-06f * ((B.ext2 + b2) + qRs);  // 2^-18
                const float rin = qRs - hw, rout = qRs + hw;
                const uint32_t occ = B.occ;
                // each child's record is loaded while the one before it is judged
                uint32_t todo = occ, c = (uint32_t)__builtin_ctz(occ | 256u);
                u32x16 nx = child_box(B, c & 7u);
                while (todo) {
                    const u32x16 x = nx;
                    todo &= todo - 1u;
                    c = (uint32_t)__builtin_ctz(todo | 256u);
                    nx = child_box(B, c & 7u);
                    const float hx = __uint_as_float(x[3]), hy = __uint_as_float(x[4]), hz = __uint_as_float(x[5]);
                    const float ex = fabsf(bx - __uint_as_float(x[0])), ey = fabsf(by - __uint_as_float(x[1]));
                    const float ez = fabsf(bz - __uint_as_float(x[2]));
                    const float mx = ex + hx, my = ey + hy, mz = ez + hz;
                    const float fx = clamp01(ex - hx), fy = clamp01(ey - hy), fz = clamp01(ez - hz);
                    const uint64_t in = m & ballot64(__builtin_fmaf(mx, mx, __builtin_fmaf(my, my, mz * mz)) <= rin);
                    const uint64_t ov = m & ~in & ~ballot64(__builtin_fmaf(fx, fx, __builtin_fmaf(fy, fy, fz * fz)) > rout);
                    if (__builtin_amdgcn_inverse_ballot_w64(in)) cnt += x[6];
                    if (ov) {
                        if (x[7] == 0) {
                            NodeRec ur;
                            auto f64 = [](uint32_t lo, uint32_t hi) { return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo)); };
                            ur.cx = f64(x[8], x[9]), ur.cy = f64(x[10], x[11]), ur.cz = f64(x[12], x[13]);
                            ur.first = x[14], ur.last = x[14] + x[6];
                            leaf_mfma(ov, __uint_as_float(x[15]), ur, true);
                        } else if (sp < kStack) {
                            s_node[w][sp] = x[7], s_mask[w][sp] = ov, s_depth[w][sp] = (uint8_t)d;
                            sp++;
                        } else {
                            overflow = 1;
                        }
                    }
                }
                continue;
            }
        }
        uint64_t inl[8], ovl[8];
        judge8(E, d, actm, inl, ovl);
        if (STATS) n_class += 8ull * __popcll(m), n_cslots += 64ull * 8;
        if constexpr (MODE == 2) {
            // lists: the children in octant order - INSIDE ranges and leaves are emitted, internal nodes wait (popped
            // last pushed first, as the reference does). ev: combos with an INSIDE or OVERLAP query; an empty
            // child changes nothing but a range list, which keeps empty INSIDE ranges (neighbor_set.hpp:84-89)
            uint32_t ev = 0;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const bool some = E.last[c] > E.first[c];
                const uint64_t im = kRanges || some ? inl[c] : 0ull, om = some ? ovl[c] : 0ull;
                if (im | om) {
                    if (lane == 0) s_inm[w][c] = im, s_leafm[w][c] = om;
                    ev |= 1u << c;
                }
            }
            ev = uniform_u32(ev);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
            for (uint32_t o = 0; o < 8; o++) {
                const uint32_t c = (E.order[o >> 2] >> (8u * (o & 3u))) & 7u;
                if (!((ev >> c) & 1u)) continue;
                const uint64_t im = uniform_u64(s_inm[w][c]), om = uniform_u64(s_leafm[w][c]);
                const uint32_t f = E.first[c], l = E.last[c];
                if (__builtin_amdgcn_inverse_ballot_w64(im)) {
                    if (kRanges) {
                        out[0] = f, out[1] = l;
                        out += 2;
                    } else {
                        for (uint32_t i = f; i < l; i++) *out++ = i;
                    }
                }
                if (om) {
                    const uint32_t gc = E.gc[c];
                    if (gc == 0) {
                        NodeRec ur;
                        ur.cx = E.ax[c & 1], ur.cy = E.ax[2 + ((c >> 1) & 1)], ur.cz = E.ax[4 + ((c >> 2) & 1)];
                        ur.first = f, ur.last = l;
                        leaf_lists(om, E.amax[c], ur);
                    } else if (sp < kStack) {
                        s_node[w][sp] = gc, s_mask[w][sp] = om, s_depth[w][sp] = (uint8_t)d;
                        sp++;
                    } else {
                        overflow = 1;
                    }
                }
            }
        } else {
            // INSIDE children first: group 0's lanes (0 .. G - 1) hold the counts
#pragma unroll
            for (int c = 0; c < 8; c++)
                if (__builtin_amdgcn_inverse_ballot_w64(inl[c] & gmask)) {
                    cnt += E.last[c] - E.first[c];
                    if (MODE == 1) ecnt++;  // NeighborSet::addRange keeps empty ranges (neighbor_set.hpp:84-89)
                }
            uint32_t leaves = 0;  // combos of the OVERLAP non-empty leaf children (bit c)
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const uint32_t f = E.first[c], l = E.last[c];
                const uint64_t ov = ovl[c] & gmask;  // ballots: uniform already
                if (ov) {
                    const uint32_t gc = E.gc[c];
                    if (gc == 0) {
                        if (l > f) {  // an empty leaf adds nothing to a count
                            if (lane == 0) s_leafm[w][c] = ov;
                            leaves |= 1u << c;
                        }
                    } else if (sp < kStack) {
                        s_node[w][sp] = gc, s_mask[w][sp] = ov, s_depth[w][sp] = (uint8_t)d;
                        sp++;
                    } else {
                        overflow = 1;
                    }
                }
            }
            // the leaves, one code copy: their records are scalar loads from E at a uniform index
            leaves = uniform_u32(leaves);  // built from ballots: the same in every lane
            if (leaves) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            while (leaves) {
                const uint32_t c = (uint32_t)__builtin_ctz(leaves);
                leaves &= leaves - 1;
                const uint64_t ov = uniform_u64(s_leafm[w][c]);
                NodeRec ur;
                ur.cx = E.ax[c & 1], ur.cy = E.ax[2 + ((c >> 1) & 1)], ur.cz = E.ax[4 + ((c >> 2) & 1)];
                ur.first = E.first[c], ur.last = E.last[c];
                if constexpr (kMfma)
                    leaf_mfma(ov, E.amax[c], ur, false);
                else if constexpr (MODE == 0)
                    leaf(ov, E.amax[c], ur);
                else
                    leaf_lists(ov, E.amax[c], ur);
            }
        }
    }
    // the S lanes of a query hold parts of its count: lanes j, j + G, ... (G >= 16)
    if constexpr (G <= 16) cnt += lane_xor<16>(cnt);
    if constexpr (G <= 32) cnt += lane_xor32(cnt);
    if (overflow && lane == 0) atomicOr(a.err, kErrStack);
    if (MODE != 2 && valid && g == 0) {
        if (a.counts) a.counts[qid] = cnt;
        const uint32_t ec = MODE == 1 ? ecnt : cnt;  // index lists: one entry per neighbour
        if (a.ecounts) a.ecounts[qid] = ec;
        if (a.ecounts64) a.ecounts64[qid] = ec;
    }
    if (STATS) {
        if (lane == 0) {
            atomicAdd(&a.stats[0], (unsigned long long)n_class);
            atomicAdd(&a.stats[1], (unsigned long long)n_test);
            atomicAdd(&a.stats[4], (unsigned long long)n_cslots);
            atomicAdd(&a.stats[5], (unsigned long long)n_tslots);
        }
        uint64_t r = n_recheck, nb = (valid && g == 0) ? cnt : 0;
        for (int off = 32; off > 0; off >>= 1) r += __shfl_xor(r, off), nb += __shfl_xor(nb, off);
        if (lane == 0) {
            if (r) atomicAdd(&a.stats[2], (unsigned long long)r);
            atomicAdd(&a.stats[3], (unsigned long long)nb);
        }
    }
}

template <int KERNEL, int ALGO, int PREC, int G, bool STATS>
__global__ __launch_bounds__(kSearchBlock) __attribute__((amdgpu_waves_per_eu(count_waves<KERNEL, ALGO, PREC>()))) void k_count(const SearchArgs a) {
    count_tile<KERNEL, ALGO, PREC, G, STATS>(a, blockIdx.x * kWaves + (threadIdx.x >> 6));
}

// Sizes (MODE 1, range lists) and fill (MODE 2) of result lists, 64 consecutive queries per wave.
template <int KERNEL, int ALGO, int PREC, bool STATS, int MODE>
__global__ __launch_bounds__(kSearchBlock) void k_lists(const SearchArgs a) {
    count_tile<KERNEL, ALGO, PREC, 64, STATS, MODE>(a, blockIdx.x * kWaves + (threadIdx.x >> 6));
}

// Work-queue form (batches): a grid of resident waves; each wave takes the next wave tile from a
// device counter (queue_next) until the device-resident tile count (queue_tiles) is reached, so the
// launch shape does not depend on how many tiles the queries made. Every wave leaves once the
// counter has passed the count.
template <int KERNEL, int ALGO, int PREC>
__global__ __launch_bounds__(kSearchBlock) __attribute__((amdgpu_waves_per_eu(count_waves<KERNEL, ALGO, PREC>()))) void k_count_queue(const SearchArgs a) {
    const uint32_t ntiles = uniform_u32(*a.queue_tiles);
    for (;;) {
        uint32_t t = 0;
        if (lane_id() == 0) t = atomicAdd(a.queue_next, 1u);
        t = readlane_u32(t, 0);
        if (t >= ntiles) return;
        count_tile<KERNEL, ALGO, PREC, 64, false>(a, t);
    }
}

template <int KERNEL, int ALGO, int PREC, bool STATS>
static void launch_count_s(const SearchArgs &a, int G, hipStream_t s) {
    const size_t tiles = ((size_t)a.nq + G - 1) / G;
    const unsigned nb = (unsigned)((tiles + kWaves - 1) / kWaves);
    if (G == 16)
        k_count<KERNEL, ALGO, PREC, 16, STATS><<<nb, kSearchBlock, 0, s>>>(a);
    else if (G == 32)
        k_count<KERNEL, ALGO, PREC, 32, STATS><<<nb, kSearchBlock, 0, s>>>(a);
    else
        k_count<KERNEL, ALGO, PREC, 64, STATS><<<nb, kSearchBlock, 0, s>>>(a);
}

// resident waves of the work-queue kernel: blocks per CU at its occupancy, times the CUs
template <int KERNEL, int ALGO, int PREC>
static unsigned group_queue_grid(size_t lds) {  // lds: always that of kGroupMaxLevels
    static unsigned cached = 0;
    if (cached) return cached;
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_group_queue<KERNEL, ALGO, PREC>, kSearchBlock, lds);
    cached = (unsigned)((cus > 0 ? cus : 256) * (per > 0 ? per : 1));
    return cached;
}
template <int KERNEL, int ALGO, int PREC>
static unsigned queue_grid() {
    static unsigned cached = 0;
    if (cached) return cached;
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_count_queue<KERNEL, ALGO, PREC>, kSearchBlock, 0);
    cached = (unsigned)((cus > 0 ? cus : 256) * (per > 0 ? per : 1));
    return cached;
}

template <int KERNEL, int ALGO, int PREC>
static void launch_count(const SearchArgs &a, int G, hipStream_t s) {
    if constexpr (ALGO != OCT_ALGO_APPROX) {
        if (a.queue_next) {  // work-queue form: 64 queries per wave tile, no counters
            k_count_queue<KERNEL, ALGO, PREC><<<queue_grid<KERNEL, ALGO, PREC>(), kSearchBlock, 0, s>>>(a);
            return;
        }
    }
    if constexpr (ALGO == OCT_ALGO_APPROX) {  // one shape: 64 queries per wave
        const unsigned nb = (unsigned)(((size_t)a.nq + 64 * kWaves - 1) / (64 * kWaves));
        if (a.stats)
            k_count<KERNEL, ALGO, PREC, 64, true><<<nb, kSearchBlock, 0, s>>>(a);
        else
            k_count<KERNEL, ALGO, PREC, 64, false><<<nb, kSearchBlock, 0, s>>>(a);
        return;
    }
    if (a.stats)
        launch_count_s<KERNEL, ALGO, PREC, true>(a, G, s);
    else
        launch_count_s<KERNEL, ALGO, PREC, false>(a, G, s);
}

template <int KERNEL, int ALGO, int PREC>
static void launch_k(const SearchArgs &a, int mode, int G, hipStream_t s) {
    if (mode == 0 && G > 0) {
        launch_count<KERNEL, ALGO, PREC>(a, G, s);
        return;
    }
    if constexpr (ALGO != OCT_ALGO_APPROX) {
        if (G > 0) {  // lists of many queries that lie together
            const unsigned nb = (unsigned)(((size_t)a.nq + 64 * kWaves - 1) / (64 * kWaves));
            if (mode == 2)
                k_lists<KERNEL, ALGO, PREC, false, 2><<<nb, kSearchBlock, 0, s>>>(a);
            else if constexpr (ALGO != OCT_ALGO_STRUCT)
                launch_count<KERNEL, ALGO, PREC>(a, 64, s);  // an index list is as long as its count
            else if (a.stats)
                k_lists<KERNEL, ALGO, PREC, true, 1><<<nb, kSearchBlock, 0, s>>>(a);
            else
                k_lists<KERNEL, ALGO, PREC, false, 1><<<nb, kSearchBlock, 0, s>>>(a);
            return;
        }
    }
    const size_t lds = (size_t)kWaves * a.levels * 64 * sizeof(uint32_t);
    if constexpr (ALGO != OCT_ALGO_APPROX) {
        if (a.queue_next) {
            k_group_queue<KERNEL, ALGO, PREC><<<group_queue_grid<KERNEL, ALGO, PREC>(lds), kSearchBlock, lds, s>>>(a);
            return;
        }
    }
    // one launch holds 2^29 queries
    for_grids(((size_t)a.nq + kGroupsPerWave * kWaves - 1) / (kGroupsPerWave * kWaves), kSearchBlock,
              [&](uint32_t block0, unsigned nb) {
                  if (mode == 0)
                      k_group<KERNEL, ALGO, PREC, 0><<<nb, kSearchBlock, lds, s>>>(a, block0);
                  else if (mode == 1)
                      k_group<KERNEL, ALGO, PREC, 1><<<nb, kSearchBlock, lds, s>>>(a, block0);
                  else
                      k_group<KERNEL, ALGO, PREC, 2><<<nb, kSearchBlock, lds, s>>>(a, block0);
              });
}

// f(kernel, algorithm, precision), as integral constants
template <class F>
static void with_variant(int kernel, int algo, int prec, F &&f) {
    auto by_prec = [&](auto K, auto A) {
        if (prec == OCT_PREC_FP32_RECHECK)
            f(K, A, std::integral_constant<int, OCT_PREC_FP32_RECHECK>{});
        else
            f(K, A, std::integral_constant<int, OCT_PREC_FP64>{});
    };
    auto by_algo = [&](auto K) {
        if (algo == OCT_ALGO_NEIGHBORS)
            by_prec(K, std::integral_constant<int, OCT_ALGO_NEIGHBORS>{});
        else if (algo == OCT_ALGO_PRUNE)
            by_prec(K, std::integral_constant<int, OCT_ALGO_PRUNE>{});
        else if (algo == OCT_ALGO_STRUCT)
            by_prec(K, std::integral_constant<int, OCT_ALGO_STRUCT>{});
        else
            by_prec(K, std::integral_constant<int, OCT_ALGO_APPROX>{});
    };
    switch (kernel) {
    case OCT_KERNEL_SPHERE: by_algo(std::integral_constant<int, OCT_KERNEL_SPHERE>{}); break;
    case OCT_KERNEL_CIRCLE: by_algo(std::integral_constant<int, OCT_KERNEL_CIRCLE>{}); break;
    case OCT_KERNEL_CUBE: by_algo(std::integral_constant<int, OCT_KERNEL_CUBE>{}); break;
    default: by_algo(std::integral_constant<int, OCT_KERNEL_SQUARE>{}); break;
    }
}

// levels that hold internal nodes: every level but the deepest
static uint32_t group_levels(const oct_ctx *ctx) {
    return ctx->n_levels > 1 ? std::min<uint32_t>(ctx->n_levels - 1, (uint32_t)kGroupMaxLevels) : 1u;
}

hipError_t radius_resident_waves(const oct_ctx *ctx, int kernel, int algo, int precision, int group, double &waves) {
    int cus = 0, per = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device);
    if (e != hipSuccess) return e;
    with_variant(kernel, algo, precision, [&](auto K, auto A, auto P) {
        constexpr int k = decltype(K)::value, al = decltype(A)::value, p = decltype(P)::value;
        if constexpr (al != OCT_ALGO_APPROX) {
            if (group == 0)
                e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_group<k, al, p, 0>, kSearchBlock,
                                                                 (size_t)kWaves * group_levels(ctx) * 64 * sizeof(uint32_t));
            else if (group == 16)
                e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_count<k, al, p, 16, false>, kSearchBlock, 0);
            else if (group == 32)
                e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_count<k, al, p, 32, false>, kSearchBlock, 0);
            else
                e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_count<k, al, p, 64, false>, kSearchBlock, 0);
        }
    });
    waves = (double)std::max(1, cus) * (double)std::max(1, per) * kWaves;
    return e;
}

hipError_t launch_radius(oct_ctx *ctx, const RadiusLaunch &L) {
    if (L.nq == 0) return hipSuccess;
    SearchArgs a;
    a.p64 = ctx->p64.p;
    a.p32 = ctx->p32.p;
    a.amax = ctx->amax.p;
    a.nodes = ctx->nodes.p;
    a.next = ctx->next.p;
    a.nbox = nullptr, a.tie_scale = 0.0, a.tight_min = a.box_scale = 0.0f;
    stage_begin(ctx, ST_SEARCH);  // a tree's first count that uses the tight boxes makes them
    double extent = 0.0;  // clouds of 1e15 and more have no boxes: their FP32 terms are checked leaf by leaf
    for (int k = 0; k < 3; k++) extent = std::max(extent, 2.0 * fabs(ctx->radii[k]));
    if (L.mode == 0 && L.group == 64 && L.kernel == OCT_KERNEL_SPHERE && L.precision == OCT_PREC_FP32_RECHECK &&
        (L.algo == OCT_ALGO_PRUNE || L.algo == OCT_ALGO_STRUCT) && !L.tile_info && !L.stats && ctx->n_total > 1 &&
        extent < 1e15 && !ctx->no_boxes) {
        const hipError_t e = launch_boxes(ctx);
        if (e != hipSuccess && e != hipErrorOutOfMemory) return e;
        double mc = 0.0;
        for (int k = 0; k < 3; k++) mc = std::max(mc, ctx->geo[66 + k]);
        if (e == hipSuccess) {
            a.nbox = ctx->nbox.p;
        } else {  // the cells are judged, and no count of this tree asks for the memory again
            (void)hipGetLastError();
            ctx->no_boxes = true;
        }
        a.box_scale = ctx->box_scale;
        a.tie_scale = mc * 1.4210854715202004e-14;                                // 2^-46
        a.tight_min = (float)std::max(1e-30, mc * mc * 8.881784197001252e-16);  // (2^-25 mc)^2
    }
    a.child = ctx->child.p;
    a.order = L.order;
    a.qidx = L.qidx;
    a.qxyz = L.qxyz;
    a.qrad = L.qrad;
    a.radius = L.radius;
    a.qrad3 = L.qrad3;
    for (int k = 0; k < 3; k++) a.r3[k] = L.radius3[k];
    a.use_r3 = L.use_r3 ? 1 : 0;
    a.remap = L.remap ? 1 : 0;
    a.approx_level = L.approx_level;
    a.approx_upper = L.approx_upper ? 1 : 0;
    a.radtab = L.radtab ? L.radtab : ctx->radtab.p;
    a.tile_info = L.tile_info;
    a.roots = L.roots;
    a.queue_tiles = L.queue_tiles;
    a.queue_next = L.queue_next;
    a.nq = (uint32_t)L.nq;
    a.counts = L.counts;
    a.ecounts = L.ecounts;
    a.ecounts64 = L.ecounts64;
    a.offsets = L.offsets;
    a.entries = L.entries;
    a.stats = L.stats;
    a.err = ctx->derr.p;
    a.levels = L.tile_info ? (uint32_t)kGroupMaxLevels : group_levels(ctx);  // a forest's depth is not known here
    with_variant(L.kernel, L.algo, L.precision, [&](auto K, auto A, auto P) {
        launch_k<decltype(K)::value, decltype(A)::value, decltype(P)::value>(a, L.mode, L.group, ctx->stream);
    });
    stage_end(ctx, ST_SEARCH);
    return hipGetLastError();
}

}  // namespace oct
