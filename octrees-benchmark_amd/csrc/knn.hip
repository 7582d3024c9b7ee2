// H6: k nearest neighbours (LinearOctree::knn, linear_octree.hpp:899-942; harness label KNNV2).
//
// Result contract: the min(n, k) points with the smallest squared FP64 distance, the distance
// evaluated exactly as distPointsSquared (linear_octree.hpp:844-851: dx = q.x - p.x, ...,
// dx*dx + dy*dy + dz*dz, no contraction), ordered by (distance, sorted index). The reference's
// heap returns the same distances; only the order inside a tie class is unspecified there.
//
// A group of S lanes serves one query (64 / S queries per wave), each with its own traversal:
//  - a node's 8 children are judged one per lane; a child waits with a lower bound of its box distance,
//    rounded down to 16 bits. The nearest waiting child of the deepest level comes next (a min over the
//    group's lanes), and a level whose nearest child is beyond the current k-th distance is dropped. The
//    bound widens every box by 2^-40 of the cloud's magnitude, which covers the FP64 rounding of node
//    centres and of points on cell faces, so pruning never drops a true neighbour;
//  - groups go down independently until each holds a leaf; then all test their leaves' points, S (or 2 S)
//    at a time, and append those not beyond the current bound to the query's buffer in LDS;
//  - a selection finds, by counting, a bound T on the distance's upper 32 bits with k to kw entries at or
//    below it (a few interpolated guesses: the count grows about linearly with the squared distance),
//    keeps those and drops the rest; T bounds the k-th distance from above. No entry is sorted until the
//    end, when the k best of the remaining few are ordered exactly. More than kw entries can share T's
//    upper bits (ties): where they would fill the buffer, an exact selection keeps the k best, and from then
//    on points are held against the k-th of them, distance and index. (Against T alone every further point of
//    a stack of duplicates is accepted, and one step in two ends in an exact selection: 100 k queries, a sixth
//    of them at a stack of 20 k points, k = 10: 27.8 ms, with the k-th 10.9;
//    without stacks 0 to 1.2 % slower for it, k = 10 to 1000.)
// Both precisions run the same FP64 distances: MI355X issues FP64 at the rate of unpacked FP32, and a
// leaf-recentred FP32 screen in front of them (16 instead of 32 bytes per point, a second load for what
// passes) was 6 - 17 % slower at every k from 1 to 1000.
#include <cfloat>
#include <type_traits>

#include "device.hpp"
#include "grid.hpp"
#include "search_common.hpp"

namespace oct {

struct KnnArgs {
    const double4 *__restrict__ p64;
    const NodeRec *__restrict__ nodes;
    const uint32_t *__restrict__ child;
    const uint32_t *__restrict__ order;
    const uint32_t *__restrict__ qidx;
    const double *__restrict__ qxyz;
    uint32_t nq, k;
    uint32_t qoff;  // all-points queries: slot s is sorted point qoff + s
    int32_t *__restrict__ idx_out;
    double *__restrict__ d2_out;
    float *__restrict__ d2f_out;
    unsigned long long *__restrict__ stats;
    uint32_t *__restrict__ err;  // device error word: kErrStack when the traversal stack was full
    // tree geometry per cloud: level radii radtab[cloud * 66 + 3 * level + axis] and the box magnitude
    // magtab[cloud * 3 + axis] = |centre| + radius; for a forest of clouds, tile_info[wave tile] =
    // cloud | valid slots << 20 and roots[cloud] (null: one cloud, root node 0)
    const double *__restrict__ radtab;
    const double *__restrict__ magtab;
    const uint32_t *__restrict__ tile_info;
    const uint32_t *__restrict__ roots;
    const uint32_t *__restrict__ kq;  // per-query k (null: k for every query); k is the row width
    const uint32_t *__restrict__ cloud_off;  // set: indices written local to the tile's cloud
    // work-queue form: device-resident wave-tile count and the zeroed counter waves take tiles from
    const uint32_t *__restrict__ queue_tiles;
    uint32_t *__restrict__ queue_next;
    uint32_t levels;  // rows of waiting children in LDS: the tree's levels
};

// Order of the results: squared distances are sums of squares (never -0), so their bit patterns order as
// the values do (a NaN after every number); ties by index.
__device__ inline bool knn_less(uint64_t da, uint32_t ia, uint64_t db, uint32_t ib) { return da < db || (da == db && ia < ib); }

// Lower bound of the squared distance from q to any point of the box c +- r, each axis widened by
// dl; the caller compares it against tau (1 + 2^-40), which covers the rounding of this sum.
__device__ inline double gap2(double q, double c, double r, double dl) {
    const double gap = fabs(q - c) - r - dl;
    return gap > 0.0 ? gap * gap : 0.0;
}

// Buffer entries per query for the size class KC (k <= KC): three times KC where KC is small, so that a
// selection is seldom needed, else twice.
constexpr int knn_cap(int kc) { return kc <= 32 ? 3 * kc : 2 * kc; }
constexpr uint32_t kKnnLeafBit = 0x80000000u;

// LDS of one wave: per level and group lane, the waiting child's bound (upper half of its float) and its
// first child, or its own index with kKnnLeafBit set for a leaf.
struct KnnLevels {
    uint32_t *node;
    uint16_t *key;
};

// One wave tile (64 / S queries) of a kNN search, run by one wave (a 64-thread block).
template <int S, int KC>
__device__ __attribute__((always_inline)) inline void knn_tile(const KnnArgs &a, const uint32_t tile, const KnnLevels lev) {
    constexpr int G = 64 / S;                // queries per wave
    constexpr int CAP = knn_cap(KC);         // buffer entries per query
    constexpr int U = S <= 16 ? 2 : 1;       // points per lane per step
    constexpr int STEP = S * U;              // points per query per step
    constexpr int ROWS = (CAP + S - 1) / S;  // buffer entries per lane
    constexpr bool kRank = KC <= 32;         // final order by counting ranks, else by a bitonic sort in LDS
    static_assert(CAP - STEP >= KC, "a step must fit after a selection");
    __shared__ uint64_t s_bd[G * CAP];
    __shared__ uint32_t s_bi[G * CAP];
    __shared__ uint64_t s_kd[G];  // with `ties`: the k-th entry of the group's last exact selection
    __shared__ uint32_t s_ki[G];
    __shared__ double s_rad[66];

    const uint32_t lane = threadIdx.x;
    const uint32_t qs = lane / S, c = lane % S, gshift = lane & ~(uint32_t)(S - 1);
    const uint32_t slot0 = tile * G;
    const uint32_t slot = slot0 + qs;
    uint32_t cloud = 0, nvt = G, root = 0;
    if (a.tile_info) {
        const uint32_t ti = uniform_u32(a.tile_info[tile]);
        cloud = ti & 0xfffffu, nvt = ti >> 20;
        root = uniform_u32(a.roots[cloud]);
    }
    ConstDouble *magp = const_doubles(a.magtab) + 3 * cloud;
    auto wsync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    wsync();
    for (uint32_t i = lane; i < 66; i += 64) s_rad[i] = a.radtab[66 * (size_t)cloud + i];
    const bool valid = slot < a.nq && qs < nvt;
    const uint32_t kw_out = a.k;  // output row width
    uint64_t *bd = s_bd + qs * CAP;
    uint32_t *bi = s_bi + qs * CAP;

    uint32_t qid = 0, k = kw_out;
    double qx = 0.0, qy = 0.0, qz = 0.0;
    if (valid) {
        qid = a.order ? a.order[slot] : slot;
        if (a.kq) k = a.kq[qid];
        if (a.qxyz) {
            qx = a.qxyz[3 * (size_t)qid], qy = a.qxyz[3 * (size_t)qid + 1], qz = a.qxyz[3 * (size_t)qid + 2];
        } else {
            const double4 p = a.p64[a.qidx ? a.qidx[qid] : a.qoff + qid];
            qx = p.x, qy = p.y, qz = p.z;
        }
    }
    // box widening per axis: 2^-40 of the magnitudes involved (cloud box and query)
    const double dlx = 0x1p-40 * (magp[0] + fabs(qx)), dly = 0x1p-40 * (magp[1] + fabs(qy));
    const double dlz = 0x1p-40 * (magp[2] + fabs(qz));

    // lanes of the own group set in a ballot; those below this lane
    auto gmask = [&](uint64_t m) -> uint64_t { return S == 64 ? m : (m >> gshift) & ((1ull << (S & 63)) - 1ull); };
    auto gcount = [&](uint64_t m) -> uint32_t {
        return S == 64 ? (uint32_t)__popcll(m) : (uint32_t)__popc((uint32_t)gmask(m));
    };
    auto gbelow = [&](uint64_t m) -> uint32_t {
        if (S == 64) return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        return (uint32_t)__popc((uint32_t)gmask(m) & ((1u << (c & 31)) - 1u));
    };
    auto hi32 = [](uint64_t b) -> uint32_t { return (uint32_t)(b >> 32); };
    auto dbits = [](double d) -> uint64_t { return (uint64_t)__double_as_longlong(d); };
    auto key_value = [](uint32_t key) -> double { return __longlong_as_double((long long)((uint64_t)key << 32)); };

    // a selection stops at k .. kw entries (an eighth more than k; a size class's own size where that bound
    // lies in between, so that the final sort stays at that size). k + k / 4 was 1 - 10 % slower.
    uint32_t kw = k + (k >> 3) + 1;
    if (kw > (uint32_t)KC && k < (uint32_t)KC) kw = KC;
    constexpr uint32_t kFresh = KC / 2 > 8 ? KC / 2 : 8;  // appended entries that are worth a new bound
    uint32_t cnt = 0, kept = 0;   // entries in the buffer; of them, after the last selection
    uint32_t T = 0xffffffffu;     // entries have upper distance bits <= T; ~0: fewer than k seen
    bool ties = false;            // an exact selection took place (the wave's groups together)
    double tau = __builtin_huge_val();      // FP64 upper bound of the k-th distance with the pruning margin
    float tauf = __builtin_huge_valf();     // the same rounded up to FP32
    uint32_t n_nodes = 0, n_test = 0, n_select = 0, n_steps = 0;

    // rank of entry (d, i) among the group's cnt entries, for every row of the buffer; entries of rank
    // below `keep` move to their rank. Afterwards the first `keep` entries are sorted.
    auto rank_sort = [&](auto rows, const uint32_t keep) {
        constexpr int R = decltype(rows)::value;
        wsync();
        uint64_t d[R];
        uint32_t ix[R], rk[R];
#pragma unroll
        for (int j = 0; j < R; j++) {
            const uint32_t t = j * S + c;
            d[j] = t < cnt ? bd[t] : ~0ull, ix[j] = t < cnt ? bi[t] : 0xffffffffu, rk[j] = 0;
        }
        for (uint32_t t = 0; ballot64(t < cnt); t++) {
            const bool in = t < cnt;
            const uint64_t dt = in ? bd[t] : ~0ull;
            const uint32_t it = in ? bi[t] : 0xffffffffu;
#pragma unroll
            for (int j = 0; j < R; j++) rk[j] += knn_less(dt, it, d[j], ix[j]) ? 1u : 0u;
        }
        wsync();
#pragma unroll
        for (int j = 0; j < R; j++)
            if ((uint32_t)(j * S) + c < cnt && rk[j] < keep) bd[rk[j]] = d[j], bi[rk[j]] = ix[j];
        wsync();
    };
    // bitonic sort of the buffer's first n entries (n a power of two) by (distance, index), two stages per
    // LDS round trip: a lane takes the 4 entries that strides s and s / 2 connect through both
    auto cx = [](uint64_t &da, uint32_t &ia, uint64_t &db, uint32_t &ib, const bool up) {
        const bool sw = up ? knn_less(db, ib, da, ia) : knn_less(da, ia, db, ib);
        const uint64_t d = sw ? db : da;
        const uint32_t i = sw ? ib : ia;
        db = sw ? da : db, ib = sw ? ia : ib;
        da = d, ia = i;
    };
    auto bitonic = [&](const uint32_t n) {
        for (uint32_t t = cnt + c; t < n; t += S) bd[t] = ~0ull, bi[t] = 0xffffffffu;
        wsync();
#pragma unroll 1
        for (uint32_t size = 2; size <= n; size <<= 1) {
            uint32_t stride = size >> 1;
#pragma unroll 1
            for (; stride >= 2; stride >>= 2) {
                const uint32_t h = stride >> 1;
#pragma unroll 1
                for (uint32_t t = c; t < n / 4; t += S) {
                    const uint32_t e0 = ((t & ~(h - 1)) << 2) | (t & (h - 1));
                    const uint32_t e1 = e0 + h, e2 = e0 + stride, e3 = e2 + h;
                    const bool up = (e0 & size) == 0;
                    uint64_t d0 = bd[e0], d1 = bd[e1], d2 = bd[e2], d3 = bd[e3];
                    uint32_t i0 = bi[e0], i1 = bi[e1], i2 = bi[e2], i3 = bi[e3];
                    cx(d0, i0, d2, i2, up);
                    cx(d1, i1, d3, i3, up);
                    cx(d0, i0, d1, i1, up);
                    cx(d2, i2, d3, i3, up);
                    bd[e0] = d0, bd[e1] = d1, bd[e2] = d2, bd[e3] = d3;
                    bi[e0] = i0, bi[e1] = i1, bi[e2] = i2, bi[e3] = i3;
                }
                wsync();
            }
            if (stride == 1) {  // an odd number of stages: the last one alone
#pragma unroll 1
                for (uint32_t t = c; t < n / 2; t += S) {
                    const uint32_t e0 = t << 1;
                    uint64_t d0 = bd[e0], d1 = bd[e0 + 1];
                    uint32_t i0 = bi[e0], i1 = bi[e0 + 1];
                    cx(d0, i0, d1, i1, (e0 & size) == 0);
                    bd[e0] = d0, bd[e0 + 1] = d1;
                    bi[e0] = i0, bi[e0 + 1] = i1;
                }
                wsync();
            }
        }
    };
    // the buffer's entries in order, the first min(cnt, k) of them exact (every lane of the wave)
    auto order_entries = [&]() {
        if (kRank) {
            constexpr int kFew = (KC + KC / 8 + 1 + S - 1) / S;  // rows that hold kw entries
            if (ballot64(cnt > (uint32_t)(kFew * S)))
                rank_sort(std::integral_constant<int, ROWS>(), k);
            else
                rank_sort(std::integral_constant<int, kFew>(), k);
        } else {
            uint32_t mx = group_reduce<64>(cnt, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
            uint32_t n = 64;
            mx = uniform_u32(mx);
            while (n < mx) n <<= 1;
            bitonic(n);
        }
        if (cnt > k) cnt = k;
    };
    auto set_bound = [&](const bool part) {  // T is valid: the k-th distance lies below (T + 1) << 32
        if (part) {
            const double ub = __longlong_as_double((long long)(((uint64_t)T + 1ull) << 32));
            tau = ub * (1.0 + 0x1p-40);
            tauf = __double2float_ru(tau);
        }
    };

    // selection, for the groups with at least k entries: T such that k .. kw entries have upper bits <= T
    // (more where they tie); the others leave the buffer
    auto select = [&]() {
        n_select++;
        wsync();
        const bool part = cnt >= k && k > 0;
        uint32_t key[ROWS];
        uint32_t mx = 0;
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const uint32_t t = j * S + c;
            key[j] = t < cnt ? hi32(bd[t]) : 0xffffffffu;
            if (t < cnt && key[j] > mx) mx = key[j];
        }
        mx = group_reduce<S>(mx, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
        // count(<= hi) = ch >= k, count(<= lo) = cl < k (lo = -1: none); keys stay below 2^31 (or a NaN's)
        uint32_t hi = mx, ch = cnt, cl = 0;
        int64_t lo = -1;
        double vlo = 0.0;
        const uint32_t target = k + ((kw - k) >> 1);
        for (uint32_t iter = 0;; iter++) {
            const bool go = part && ch > kw && (int64_t)hi - lo > 1;
            if (!ballot64(go)) break;
            const double vhi = key_value(hi);
            uint32_t mid = hi32(dbits(vlo + (vhi - vlo) * (double)((float)(target - cl) * __builtin_amdgcn_rcpf((float)(ch - cl)))));
            if (iter >= 6 || !((int64_t)mid > lo && mid < hi)) mid = (uint32_t)(lo + ((int64_t)hi - lo) / 2);
            uint32_t nle = 0;
#pragma unroll
            for (int j = 0; j < ROWS; j++) nle += key[j] <= mid ? 1u : 0u;
            nle = group_reduce<S>(nle, [](uint32_t x, uint32_t y) { return x + y; });
            if (go) {
                if (nle >= k)
                    hi = mid, ch = nle;
                else
                    lo = (int64_t)mid, cl = nle, vlo = key_value(mid);
            }
        }
        if (part) T = hi;
        // entries at or below T move to the front (towards lower slots only, row by row)
        if (ballot64(part && ch < cnt)) {
            uint32_t base = 0;
#pragma unroll
            for (int j = 0; j < ROWS; j++) {
                const uint32_t t = j * S + c;
                const bool keep = t < cnt && key[j] <= T;
                const uint64_t m = ballot64(keep);
                uint64_t d = 0;
                uint32_t ix = 0;
                if (keep) d = bd[t], ix = bi[t];
                wsync();
                if (keep) {
                    const uint32_t pos = base + gbelow(m);
                    bd[pos] = d, bi[pos] = ix;
                }
                base += gcount(m);
                wsync();
            }
            cnt = base;
        }
        set_bound(part);
        if (ballot64(cnt > (uint32_t)(CAP - STEP))) {  // ties fill the buffer: keep exactly the k best
            order_entries();
            wsync();
            if (c == 0) {
                if (part)
                    s_kd[qs] = bd[k - 1], s_ki[qs] = bi[k - 1];
                else if (!ties)
                    s_kd[qs] = ~0ull, s_ki[qs] = 0xffffffffu;
            }
            ties = true;
            wsync();
        }
        kept = cnt;
    };

    // appends the accepted points of a step; accepted lanes: upper distance bits <= T
    auto append = [&](const bool acc, const uint64_t d, const uint32_t id) {
        const uint64_t m = ballot64(acc);
        if (acc) {
            const uint32_t pos = cnt + gbelow(m);
            bd[pos] = d, bi[pos] = id;
        }
        cnt += gcount(m);
    };

    // levels with waiting children (the same in the group's lanes); levels at which this lane's child waits
    uint32_t lvl = 0, pend = 0;
    bool overflow = false;
    uint32_t i = 0, e = 0;  // the group's leaf: points left to test
    wsync();
    auto judge = [&](const bool act, const uint32_t fc, const uint32_t L) {
        // children fc .. fc + 7 (level L) of a node of the group's query, one per lane c < 8
        bool wait = false;
        uint32_t ent = 0, lbits = 0;
        if (act && c < 8) {
            const uint32_t node = fc + c;
            const NodeRec nr = a.nodes[node];
            const uint32_t gc = a.child[node];
            const double lb = (gap2(qx, nr.cx, s_rad[3 * L], dlx) + gap2(qy, nr.cy, s_rad[3 * L + 1], dly)) +
                              gap2(qz, nr.cz, s_rad[3 * L + 2], dlz);
            wait = nr.last > nr.first && !(lb > tau);
            ent = gc ? gc : (node | kKnnLeafBit);
            lbits = __float_as_uint((float)lb);  // rounded to nearest: one ulp less is a lower bound
            lbits -= lbits ? 1u : 0u;
        }
        if (wait) {
            if (L < a.levels) {
                lev.node[(L * G + qs) * 8 + c] = ent;
                lev.key[(L * G + qs) * 8 + c] = (uint16_t)(lbits >> 16);
                pend |= 1u << L;
            } else {
                overflow = true;  // below the tree's last level: cannot happen
            }
        }
        if (act && gmask(ballot64(wait))) lvl |= 1u << L;
    };
    {
        const uint32_t c0 = uniform_u32(a.child[root]);
        if (c0 == 0) {
            if (valid) i = a.nodes[root].first, e = a.nodes[root].last, n_nodes += c == 0 ? 1u : 0u;
        } else {
            judge(valid, c0, 1);
            if (c == 0 && valid) n_nodes += 8;
        }
    }
    for (;;) {
        // Groups without points take their nearest waiting child until three quarters of the groups that go on
        // have points; then those test them until more groups wait than test. (Every group until all had a leaf,
        // and until all were done with it: 72 pops and 44 steps per wave at k = 10 on the tile.)
        for (;;) {
            const bool go = i >= e && lvl != 0;
            const uint64_t wait = ballot64(go);
            if (!wait || __popcll(ballot64(i < e)) >= 3 * __popcll(wait)) break;
            wsync();
            const uint32_t L = go ? 31u - (uint32_t)__clz(lvl) : 0u;
            const bool mine = go && ((pend >> L) & 1u);
            uint32_t key = mine ? ((uint32_t)lev.key[(L * G + qs) * 8 + (c & 7u)] << 16) | c : 0xffffffffu;
            key = group_reduce<S>(key, [](uint32_t x, uint32_t y) { return x < y ? x : y; });
            const bool far = __uint_as_float(key & 0xffff0000u) > tauf;  // and so are the others of the level
            const uint32_t oct = key & 7u;
            const bool take = go && !far;
            const uint32_t ent = take ? lev.node[(L * G + qs) * 8 + oct] : 0u;
            if (mine && (far || c == oct)) pend &= ~(1u << L);
            if (go && !gmask(ballot64(mine && !far && c != oct))) lvl &= ~(1u << L);  // nothing waits at L any more
            const bool lf = take && (ent & kKnnLeafBit) != 0;
            if (lf) {
                const NodeRec &nr = a.nodes[ent & ~kKnnLeafBit];
                i = nr.first, e = nr.last;
                n_nodes += c == 0 ? 1u : 0u;
            }
            const bool down = take && !lf;
            if (ballot64(down)) {
                n_nodes += down && c == 0 ? 8u : 0u;
                judge(down, ent, L + 1);
            }
        }
        // leaf points, STEP at a time; selections in between: a first bound as soon as k points are known, a
        // new one when enough points came in or no step's points fit, and one at the end
        const bool last = ballot64(i < e) == 0;  // every traversal is done
        for (;;) {
            const bool full = i < e ? cnt + STEP > (uint32_t)CAP
                                    : (last ? cnt > kw : cnt >= k && (T == 0xffffffffu || cnt - kept >= kFresh));
            if (ballot64(full)) select();
            const uint64_t test = ballot64(i < e);
            if (!test || __popcll(ballot64(i >= e && lvl != 0)) > __popcll(test)) break;
            n_steps++;
            bool acc[U];
            uint64_t d[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t id = i + (uint32_t)(u * S) + c;
                acc[u] = id < e;
                d[u] = 0;
                if (i < e) {  // reads up to 2 S - 1 points past the range: the sorted clouds are padded
                    const double4 p = a.p64[id];
                    const double dx = qx - p.x, dy = qy - p.y, dz = qz - p.z;
                    d[u] = dbits(dx * dx + dy * dy + dz * dz);
                    n_test += acc[u] ? 1u : 0u;
                    acc[u] = acc[u] & (hi32(d[u]) <= T);
                }
            }
            if (ties) {
                const uint64_t kd = s_kd[qs];
                const uint32_t ki = s_ki[qs];
#pragma unroll
                for (int u = 0; u < U; u++) acc[u] = acc[u] & knn_less(d[u], i + (uint32_t)(u * S) + c, kd, ki);
            }
#pragma unroll
            for (int u = 0; u < U; u++) append(acc[u], d[u], i + (uint32_t)(u * S) + c);
            i = i < e ? i + STEP : i;
        }
        if (last) break;
    }
    order_entries();
    if (ballot64(overflow) && lane == 0) atomicOr(a.err, kErrStack);

    wsync();
    if (valid) {
        const uint32_t off = a.cloud_off ? a.cloud_off[cloud] : 0u;  // the tile's cloud holds every neighbour
        for (uint32_t t = c; t < kw_out; t += S) {
            const bool have_t = t < cnt;
            const double d = have_t ? __longlong_as_double((long long)bd[t]) : 0.0;
            a.idx_out[(size_t)qid * kw_out + t] = have_t ? (int32_t)(bi[t] - off) : -1;
            if (a.d2_out) a.d2_out[(size_t)qid * kw_out + t] = have_t ? d : __builtin_nan("");
            if (a.d2f_out) a.d2f_out[(size_t)qid * kw_out + t] = have_t ? (float)d : __builtin_nanf("");
        }
    }
    if (a.stats) {
        uint64_t found = (valid && c == 0) ? cnt : 0, sn = n_nodes, st = n_test;
        for (int off = 32; off > 0; off >>= 1) {
            sn += __shfl_xor(sn, off);
            st += __shfl_xor(st, off);
            found += __shfl_xor(found, off);
        }
        if (lane == 0) {
            atomicAdd(&a.stats[0], (unsigned long long)sn);
            atomicAdd(&a.stats[1], (unsigned long long)st);
            atomicAdd(&a.stats[3], (unsigned long long)found);
            atomicAdd(&a.stats[4], (unsigned long long)n_select);  // wave-wide selections
            atomicAdd(&a.stats[5], (unsigned long long)n_steps);   // wave-wide leaf steps
        }
    }
}

// dynamic LDS of one wave: rows for `levels` levels
template <int S>
constexpr size_t knn_lds(uint32_t levels) {
    return (size_t)levels * (64 / S) * 8 * (sizeof(uint32_t) + sizeof(uint16_t));
}
template <int S>
__device__ inline KnnLevels knn_levels(const KnnArgs &a) {
    extern __shared__ uint32_t s_lev[];
    return KnnLevels{s_lev, reinterpret_cast<uint16_t *>(s_lev + (size_t)a.levels * (64 / S) * 8)};
}

template <int S, int KC>
__global__ __launch_bounds__(64) void k_knn(const KnnArgs a, const uint32_t tile0) {
    knn_tile<S, KC>(a, tile0 + blockIdx.x, knn_levels<S>(a));
}

// Work-queue form (batches): a grid of resident waves; each takes the next wave tile from a device
// counter (queue_next) until the device-resident tile count (queue_tiles) is reached. Every wave
// leaves once the counter has passed the count.
template <int S, int KC>
__global__ __launch_bounds__(64) void k_knn_queue(const KnnArgs a) {
    const uint32_t ntiles = uniform_u32(*a.queue_tiles);
    for (;;) {
        uint32_t t = 0;
        if (lane_id() == 0) t = atomicAdd(a.queue_next, 1u);
        t = readlane_u32(t, 0);
        if (t >= ntiles) return;
        knn_tile<S, KC>(a, t, knn_levels<S>(a));
    }
}

template <int S, int KC>
static unsigned knn_queue_grid() {
    static unsigned cached = 0;
    if (cached) return cached;
    int dev = 0, cus = 0, per = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_knn_queue<S, KC>, 64, knn_lds<S>(kMaxDepth + 1));
    cached = (unsigned)((cus > 0 ? cus : 256) * (per > 0 ? per : 1));
    return cached;
}

template <int S, int KC>
static void launch_sk(const KnnArgs &a, hipStream_t s) {
    const size_t lds = knn_lds<S>(a.levels);
    if (a.queue_next) {
        k_knn_queue<S, KC><<<knn_queue_grid<S, KC>(), 64, lds, s>>>(a);
        return;
    }
    // one launch holds 2^29 queries of 8 lanes, 2^26 of 64
    for_grids(((size_t)a.nq + (64 / S) - 1) / (64 / S), 64,
              [&](uint32_t tile0, unsigned nb) { k_knn<S, KC><<<nb, 64, lds, s>>>(a, tile0); });
}

// buffer size class of k (entries per query kept between selections)
static int knn_kc(uint32_t k) {
    int kc = 16;
    while ((uint32_t)kc < k) kc <<= 1;
    return kc;
}

// lanes-per-query shapes of each size class, default first
int knn_lane_options(uint32_t k, int out[3]) {
    switch (knn_kc(k)) {
        case 16: case 32: out[0] = 8; return 1;
        case 64: out[0] = 16, out[1] = 8; return 2;
        case 128: out[0] = 32, out[1] = 16; return 2;
        case 256: out[0] = 64, out[1] = 32; return 2;
        default: out[0] = 64; return 1;
    }
}
// the shape that runs a requested number of lanes per query (0: not offered for this k): the smaller
// requests a class accepts run its smallest shape
int knn_shape_lanes(uint32_t k, int lanes) {
    const int kc = knn_kc(k);
    if (lanes != 2 && lanes != 4 && lanes != 8 && lanes != 16 && lanes != 32 && lanes != 64) return 0;
    if (kc <= 32) return lanes <= 8 ? 8 : 0;
    if (kc == 64) return lanes < 4 || lanes > 16 ? 0 : (lanes == 16 ? 16 : 8);
    if (kc == 128) return lanes < 8 || lanes > 32 ? 0 : (lanes == 32 ? 32 : 16);
    if (kc == 256) return lanes < 16 ? 0 : (lanes == 64 ? 64 : 32);
    return lanes == 64 ? 64 : 0;
}

static bool launch_knn_shape(const KnnArgs &a, int kc, int lanes, hipStream_t s) {
#define OCT_KNN_CASE(KCV, SV)                     \
    if (kc == KCV && lanes == SV) {               \
        launch_sk<SV, KCV>(a, s);                 \
        return true;                              \
    }
    OCT_KNN_CASE(16, 8) OCT_KNN_CASE(32, 8)
    OCT_KNN_CASE(64, 8) OCT_KNN_CASE(64, 16)
    OCT_KNN_CASE(128, 16) OCT_KNN_CASE(128, 32)
    OCT_KNN_CASE(256, 32) OCT_KNN_CASE(256, 64)
    OCT_KNN_CASE(512, 64) OCT_KNN_CASE(1024, 64)
#undef OCT_KNN_CASE
    return false;
}

hipError_t launch_knn(oct_ctx *ctx, const KnnLaunch &L, std::string &err) {
    const size_t nq = L.nq;
    const uint32_t k = L.k;
    if (k > 1024) {
        err = "knn: k above 1024 is not supported";
        return hipErrorInvalidValue;
    }
    if (nq > 0xffffffffull) {
        err = "knn: more than 2^32 - 1 queries in one call";
        return hipErrorInvalidValue;
    }
    if (nq == 0 || k == 0) return hipSuccess;
    KnnArgs a;
    a.p64 = ctx->p64.p;
    a.nodes = ctx->nodes.p;
    a.child = ctx->child.p;
    a.order = L.order;
    a.qidx = L.qidx;
    a.qxyz = L.qxyz;
    a.nq = (uint32_t)nq;
    a.k = k;
    a.qoff = L.qoff;
    a.idx_out = L.idx;
    a.d2_out = L.d2;
    a.d2f_out = L.d2f;
    a.stats = L.stats;
    a.err = ctx->derr.p;
    a.radtab = ctx->radtab.p;
    a.magtab = ctx->radtab.p + 66;  // the context's magnitudes follow its level radii
    a.tile_info = L.tile_info;
    a.roots = L.roots;
    a.kq = L.kq;
    a.cloud_off = L.cloud_off;
    a.queue_tiles = L.queue_tiles;
    a.queue_next = L.queue_next;
    if (L.radtab) a.radtab = L.radtab, a.magtab = L.magtab;
    const uint32_t kcls = L.kq && L.kclass ? L.kclass : k;  // selection size class of the launch
    int opts[3];
    knn_lane_options(kcls, opts);
    const int lanes = L.lanes > 0 ? knn_shape_lanes(kcls, L.lanes) : opts[0];
    // rows of waiting children: levels 1 .. the deepest (a forest's depth is known on the device only)
    a.levels = L.roots ? kMaxDepth + 1 : (ctx->n_levels > 1 ? ctx->n_levels : 1u);
    stage_begin(ctx, ST_KNN);
    if (!launch_knn_shape(a, knn_kc(kcls), lanes, ctx->stream)) {
        err = "knn: lanes per query not offered for this k";
        return hipErrorInvalidValue;
    }
    stage_end(ctx, ST_KNN);
    return hipGetLastError();
}

}  // namespace oct
