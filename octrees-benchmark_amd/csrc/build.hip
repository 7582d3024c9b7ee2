// H4: linear-octree build on gfx950.
//
// The reference grows a cornerstone leaf array by rounds of split decisions (linear_octree.hpp:
// 151-333, 458-489), then derives the level-ordered node arrays (offsets, internalRanges, centers)
// by prefix sort, linking and recursion (:336-565). Starting from the root, its merges never fire,
// so its tree is the canonical one: a node splits iff it holds more than maxPointsLeaf points and
// its level is below 21, and nodes are numbered level by level, in key order within a level.
//
// This build produces those arrays directly, top-down, one level per step:
//   level l nodes -> (flag = count > M && l < 21) -> exclusive scan of flags -> children of the
//   flagged nodes are the next level, in key order, at indices levelStart[l+1] + 8 * rank + octant.
// A child's point range comes from two binary searches of the sorted keys inside its parent's
// range (the reference's lower_bound counting, :317-321); its FP64 centre is getCenter
// (point_encoder.hpp:517-539) evaluated in the reference's operation order.
// A last pass writes the leaf-recentred FP32 copy of the cloud used by the FP32 searches.
#include <cfloat>
#include <algorithm>

#include "tree_common.hpp"

namespace oct {

struct BuildGeom {
    double boxmin[3];
    double hl[3];
    double rad[22][3];
    int encoder;
};

__device__ inline void write_node(NodeRec *__restrict__ nodes, uint64_t *__restrict__ nkey, uint32_t u, uint64_t key,
                                  uint32_t level, uint32_t first, uint32_t last, const BuildGeom &g) {
    put_node(nodes, nkey, u, key, level, first, last, g.encoder, g.boxmin, g.hl, g.rad[level]);
}

__global__ void k_root(NodeRec *nodes, uint64_t *nkey, uint32_t *flags, uint32_t n, uint32_t max_leaf, BuildGeom g) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        write_node(nodes, nkey, 0, 0ull, 0, 0, n, g);
        flags[0] = (n > max_leaf) ? 1u : 0u;
    }
}

// Nodes of level `level` (indices [ls, le)), 8 lanes each. Flagged nodes write their 8 children.
__global__ __launch_bounds__(256) void k_children(const uint64_t *__restrict__ keys, NodeRec *__restrict__ nodes,
                                                 uint64_t *__restrict__ nkey, uint32_t *__restrict__ child,
                                                 const uint32_t *__restrict__ flags, const uint32_t *__restrict__ rank,
                                                 uint32_t *__restrict__ next_flags, uint32_t ls, uint32_t le, uint32_t level,
                                                 uint32_t max_leaf, BuildGeom g) {
    // 8 lanes per node (lane k: child k); a node's lanes leave or stay together
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t i = t >> 3;
    const uint32_t k = (uint32_t)(t & 7u);
    if (i >= le - ls) return;
    const uint32_t u = ls + (uint32_t)i;
    if (!flags[i]) {
        if (k == 0) child[u] = 0;
        return;
    }
    const uint32_t cb = le + 8u * rank[i];
    if (k == 0) child[u] = cb;
    const NodeRec pr = nodes[u];
    const uint64_t pkey = nkey[u];
    const uint32_t cl = level + 1;
    const uint64_t step = node_range(cl);
    // child k ends where the keys reach child k + 1's prefix; it starts where child k - 1 ends (the
    // search over the whole parent range finds the same index as one starting at child k's start)
    const uint32_t hi = (k == 7) ? pr.last : lower_bound_keys(keys, pr.first, pr.last, pkey + (uint64_t)(k + 1) * step);
    const uint32_t prev = __shfl_up(hi, 1, 8);
    const uint32_t lo = (k == 0) ? pr.first : prev;
    write_node(nodes, nkey, cb + k, pkey + (uint64_t)k * step, cl, lo, hi, g);
    next_flags[cb - le + k] = (hi - lo > max_leaf && cl < kMaxDepth) ? 1u : 0u;
}

// Leaf-recentred FP32 coordinates, kRecentreLanes lanes per node (recentre_leaf); internal nodes'
// groups leave at once.
__global__ __launch_bounds__(256) void k_recentre(const double4 *__restrict__ p64, const NodeRec *__restrict__ nodes,
                                                 const uint32_t *__restrict__ child, uint32_t n_total, float4 *__restrict__ p32,
                                                 float *__restrict__ amax) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t u = t / kRecentreLanes;
    const uint32_t g = (uint32_t)(t % kRecentreLanes);
    if (u >= n_total) return;
    if (child[u] != 0) return;
    const float m = recentre_leaf<kRecentreLanes>(p64, nodes[u], g, p32);
    if (g == 0) amax[u] = m;
}

// Per internal node u: its children regrouped by corner bits, 8 lanes per node (node_ext_child).
struct LevelTable {
    uint32_t start[kMaxDepth + 3];
};
__global__ __launch_bounds__(256) void k_node_ext(const NodeRec *__restrict__ nodes, const uint64_t *__restrict__ nkey,
                                                 const uint32_t *__restrict__ child, const float *__restrict__ amax,
                                                 uint32_t n_total, int encoder, LevelTable lt, NodeExt *__restrict__ ext) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t u = t >> 3;
    if (u >= n_total) return;
    const uint32_t fc = child[u];
    if (fc == 0) return;
    uint32_t level = 0;
    while (level + 1 < kMaxDepth + 2 && lt.start[level + 1] <= u) level++;
    node_ext_child(nodes, nkey, child, amax, fc, (uint32_t)(t & 7u), level, encoder, ext + ((fc - 1) >> 3));
}

// ---- device-driven level loop: no host round trip between levels
//
// Each level is one launch that takes the level's node range [ls, le) from ctl[l] (written by the level
// above). k_level_step walks the level in tiles of 32 to 256 nodes (dynamic tile ids; 32 nodes are one
// round of 8 lanes each, so the top levels' long searches run side by side, 256 keep the tile count of
// large levels low): it ranks a tile's split flags with ballots, takes the tile's offset from a chained
// scan over the tiles (decoupled look-back in which one wave reads 64 predecessor tiles per step, bounded
// spins), points every node at its first child (0 = leaf) and builds the children of the split nodes, 8
// lanes per node; the last tile writes ctl[l + 1]. Levels past the last one find an empty range and return (about 2.5 us each), so the host
// enqueues all of them and reads the level table back once. The node arrays are sized up front; a level
// that would outgrow them raises an error bit, and the host then runs the level loop with growing arrays
// instead. Two launches per level for the first 13 levels, and the host loop for anything deeper, took
// 0.9 ms of a 120 k-point frame whose duplicates reach below level 12.
constexpr uint32_t kLvlTileMax = 256, kLvlTileMin = 32;
constexpr size_t kLvlTiles = 2048;  // tiles of a level beyond which they grow
// nodes per tile of a level of at most nmax nodes
static uint32_t level_tile(size_t nmax) {
    uint32_t t = kLvlTileMin;
    while (t < kLvlTileMax && nmax > kLvlTiles * t) t *= 2;
    return t;
}
constexpr uint32_t kLvlAgg = 1u << 30, kLvlInc = 2u << 30, kLvlMask = (1u << 30) - 1u, kLvlSpin = 1u << 24;
constexpr uint32_t kLvlErrSpin = 1u, kLvlErrCap = 2u;
constexpr int kLvlCount = kMaxDepth + 1;  // levels 0 .. 21 (level 21 nodes never split)

struct LevelCtl {
    uint32_t ls, le;
};

// root, level table (level 0 = the root, every other level empty until its parent level fills it),
// zero look-back words, tile counters and error word
__global__ __launch_bounds__(256) void k_level_init(NodeRec *nodes, uint64_t *nkey, uint32_t *flags, uint32_t n,
                                                    uint32_t max_leaf, BuildGeom g, LevelCtl *ctl,
                                                    uint32_t *__restrict__ lookback, size_t nlook,
                                                    uint32_t *__restrict__ counters, uint32_t *__restrict__ err,
                                                    uint32_t *__restrict__ total) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = t; i < nlook; i += stride) lookback[i] = 0u;
    if (t == 0) *total = 0u;
    if (t < (size_t)kLvlCount) counters[t] = 0u;
    if (t <= (size_t)kLvlCount) ctl[t] = t == 0 ? LevelCtl{0u, 1u} : LevelCtl{0u, 0u};
    if (t == 0) {
        write_node(nodes, nkey, 0, 0ull, 0, 0, n, g);
        flags[0] = (n > max_leaf) ? 1u : 0u;
        *err = 0u;
    }
}

__global__ __launch_bounds__(256) void k_level_step(const uint64_t *__restrict__ keys, NodeRec *__restrict__ nodes,
                                                    uint64_t *__restrict__ nkey, uint32_t *__restrict__ child,
                                                    uint32_t *__restrict__ flags, LevelCtl *__restrict__ ctl, uint32_t level,
                                                    uint32_t *__restrict__ lookback, uint32_t *__restrict__ tile_counter,
                                                    uint32_t tile_nodes, uint32_t cap, uint32_t max_leaf, BuildGeom g,
                                                    uint32_t *__restrict__ err, uint32_t *__restrict__ total) {
    __shared__ uint32_t s_w[4], s_tile, s_prefix, s_u[kLvlTileMax];
    const LevelCtl L = ctl[level];
    if (L.le <= L.ls) return;
    const uint32_t ntiles = (L.le - L.ls + tile_nodes - 1) / tile_nodes;
    if (blockIdx.x >= ntiles) return;  // the others claim every tile (a claim is a serialised atomic, ~12 ns)
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t cl = level + 1, k = tid & 7u;
    const uint64_t step = node_range(cl);
    for (;;) {
        if (tid == 0) s_tile = atomicAdd(tile_counter, 1u);
        __syncthreads();
        const uint32_t tile = s_tile;
        if (tile >= ntiles) break;
        const uint32_t u = L.ls + tile * tile_nodes + tid;
        const bool mine = tid < tile_nodes && u < L.le;
        const bool f = mine && flags[u] != 0;
        const uint64_t m = ballot64(f);
        if (lane == 0) s_w[w] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t j = (uint32_t)__popcll(m & lanemask_lt()), tot = 0;  // rank of the node in the tile; split nodes
#pragma unroll
        for (uint32_t ww = 0; ww < 4; ww++) {
            const uint32_t x = s_w[ww];
            j += ww < w ? x : 0u;
            tot += x;
        }
        if (f) s_u[j] = u;
        if (w == 0) {  // chained scan over the tiles: wave 0 looks back 64 tiles per step
            uint32_t excl = 0;
            if (tile == 0) {
                if (lane == 0) store_flag(&lookback[0], kLvlInc | tot);
            } else {
                if (lane == 0) store_flag(&lookback[tile], kLvlAgg | tot);
                int64_t base = (int64_t)tile - 1;  // lane i reads tile base - i (before tile 0: an empty prefix)
                uint32_t spins = 0;
                for (;;) {
                    const int64_t t = base - (int64_t)lane;
                    const uint32_t x = t >= 0 ? load_flag(&lookback[t]) : kLvlInc;
                    const uint64_t inc = ballot64((x >> 30) == 2u), wait = ballot64((x >> 30) == 0u);
                    const uint32_t first = inc ? (uint32_t)__builtin_ctzll(inc) : 64u;  // nearest inclusive prefix
                    const uint64_t need = first >= 63u ? ~0ull : ((2ull << first) - 1ull);
                    if (wait & need) {  // a tile up to it has published nothing yet
                        if (++spins > kLvlSpin) {
                            if (lane == 0) atomicOr(err, kLvlErrSpin);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                        continue;
                    }
                    uint32_t v = lane <= first ? (x & kLvlMask) : 0u;
#pragma unroll
                    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
                    excl += v;
                    if (first < 64u) break;
                    base -= 64;
                }
                if (lane == 0) store_flag(&lookback[tile], kLvlInc | ((excl + tot) & kLvlMask));
            }
            if (lane == 0) {
                s_prefix = excl;
                if (tile == ntiles - 1) {  // the level's split count: the next level's range
                    const uint64_t nle = (uint64_t)L.le + 8ull * (excl + tot);
                    if (nle <= cap) {
                        ctl[cl] = LevelCtl{L.le, (uint32_t)nle};
                        // no node splits, or the children are the deepest level's: the tree is complete
                        if (excl + tot == 0 || cl == kMaxDepth) *total = (uint32_t)nle;
                    } else {
                        ctl[cl] = LevelCtl{L.le, L.le};
                        atomicOr(err, kLvlErrCap);
                    }
                }
            }
        }
        __syncthreads();
        const uint32_t prefix = s_prefix;
        if (mine) child[u] = f ? L.le + 8u * (prefix + j) : 0u;
        // the tile's split nodes, 8 lanes each: lane k finds child k's end and takes its start from lane k - 1
        // (a search over the whole parent range finds the same index as one from the child's start)
        for (uint32_t q = tid >> 3; q < tot; q += 32) {
            const uint32_t pu = s_u[q];
            const uint64_t cb = (uint64_t)L.le + 8ull * (prefix + q);
            if (cb + 8u > cap) {  // the node's 8 lanes move together
                if (k == 0) atomicOr(err, kLvlErrCap);
                continue;
            }
            const NodeRec pr = nodes[pu];
            const uint64_t pkey = nkey[pu];
            const uint32_t hi = (k == 7) ? pr.last : lower_bound_keys(keys, pr.first, pr.last, pkey + (uint64_t)(k + 1) * step);
            const uint32_t prev = __shfl_up(hi, 1, 8);
            const uint32_t lo = (k == 0) ? pr.first : prev;
            write_node(nodes, nkey, (uint32_t)cb + k, pkey + (uint64_t)k * step, cl, lo, hi, g);
            flags[cb + k] = (hi - lo > max_leaf && cl < kMaxDepth) ? 1u : 0u;
            if (cl == kMaxDepth) child[cb + k] = 0u;  // no step visits the deepest level
        }
        if (gridDim.x >= ntiles) break;  // one tile per workgroup
        __syncthreads();  // the next tile rewrites the shared lists
    }
}

// k_recentre / k_node_ext over a node count read from the device (the level loop's total), launched
// with grids for the node capacity (surplus workgroups return at once: cheaper than grid-stride loops
// here, 0.55 + 0.15 against 0.59 + 0.17 ms at 2.06 M nodes of 3.1 M); k_recentre_dev also writes the
// offsets sentinel child[total] = 0.
__global__ __launch_bounds__(256) void k_recentre_dev(const double4 *__restrict__ p64, const NodeRec *__restrict__ nodes,
                                                     uint32_t *__restrict__ child, const uint32_t *__restrict__ total,
                                                     float4 *__restrict__ p32, float *__restrict__ amax) {
    const uint32_t n_total = *total;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) child[n_total] = 0u;
    const size_t u = t / kRecentreLanes;
    const uint32_t g = (uint32_t)(t % kRecentreLanes);
    if (u >= n_total) return;
    if (child[u] != 0) return;
    const float m = recentre_leaf<kRecentreLanes>(p64, nodes[u], g, p32);
    if (g == 0) amax[u] = m;
}

__global__ __launch_bounds__(256) void k_node_ext_dev(const NodeRec *__restrict__ nodes, const uint64_t *__restrict__ nkey,
                                                     const uint32_t *__restrict__ child, const float *__restrict__ amax,
                                                     const uint32_t *__restrict__ total, const LevelCtl *__restrict__ ctl,
                                                     int encoder, NodeExt *__restrict__ ext) {
    __shared__ LevelCtl s_ctl[kLvlCount];
    if (threadIdx.x < (uint32_t)kLvlCount) s_ctl[threadIdx.x] = ctl[threadIdx.x];
    __syncthreads();
    const uint32_t n_total = *total;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t u = t >> 3;
    if (u >= n_total) return;
    const uint32_t fc = child[u];
    if (fc == 0) return;
    uint32_t level = 0;
    for (uint32_t l = 0; l < (uint32_t)kLvlCount; l++)
        if (s_ctl[l].ls <= u && u < s_ctl[l].le) level = l;
    node_ext_child(nodes, nkey, child, amax, fc, (uint32_t)(t & 7u), level, encoder, ext + ((fc - 1) >> 3));
}

// The box of every leaf's points relative to the leaf's centre, kRecentreLanes lanes per leaf: the FP32
// coordinates' extremes, widened by their rounding. A leaf is bad where a point's FP32 form overflows, and where a
// point lies outside the leaf's cell: keys of a box smaller than the cloud clamp the points beyond it into the edge
// cells, and the keys of an already sorted cloud are the caller's. The reference counts an INSIDE cell's points
// unseen and drops an OUTSIDE cell's, so such points count by their cell and not by where they are. slack: 2^-49 of
// the largest coordinate, several times the rounding of the keys and the cells' centres and small against the ties
// that the counts resolve by the walk from the root (tie_scale, 2^-46). The FP32 extremes settle almost every leaf;
// one whose points reach its faces to FP32's last bit is looked at in FP64.
__global__ __launch_bounds__(256) void k_leaf_box(const double4 *__restrict__ p64, const float4 *__restrict__ p32,
                                                 const NodeRec *__restrict__ nodes, const uint32_t *__restrict__ child,
                                                 const float *__restrict__ amax, const double *__restrict__ radtab,
                                                 LevelTable lt, double slack, uint32_t n_total, PointBox *__restrict__ pbox) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t u = t / kRecentreLanes;
    const uint32_t g = (uint32_t)(t % kRecentreLanes);
    if (u >= n_total || child[u] != 0) return;
    const uint32_t first = nodes[u].first, last = nodes[u].last;
    float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX};  // lo, -hi
    for (uint32_t i = first + g; i < last; i += kRecentreLanes) {
        const float4 p = p32[i];
        v[0] = fminf(v[0], p.x), v[1] = fminf(v[1], p.y), v[2] = fminf(v[2], p.z);
        v[3] = fminf(v[3], -p.x), v[4] = fminf(v[4], -p.y), v[5] = fminf(v[5], -p.z);
    }
    for (int off = kRecentreLanes / 2; off > 0; off >>= 1)
        for (int a = 0; a < 6; a++) v[a] = fminf(v[a], __shfl_xor(v[a], off));
    uint32_t level = 0, out = 0;
    while (level + 1 < kMaxDepth + 2 && lt.start[level + 1] <= u) level++;
    if (last > first) {
        double room[3];
        bool in = true;
        for (int a = 0; a < 3; a++) {
            room[a] = radtab[3 * level + a] + slack;
            // |p - c| <= e (1 + 2^-24) + 2^-150, e the largest |fl32(p - c)|
            const double e = fmax(-(double)v[a], -(double)v[3 + a]);
            in = in && e * (1.0 + 0x1p-23) + 0x1p-149 <= room[a];
        }
        if (!in) {  // the leaf's lanes together
            const NodeRec nr = nodes[u];
            for (uint32_t i = first + g; i < last; i += kRecentreLanes) {
                const double4 p = p64[i];
                out |= fabs(p.x - nr.cx) <= room[0] && fabs(p.y - nr.cy) <= room[1] && fabs(p.z - nr.cz) <= room[2] ? 0u : 1u;
            }
            for (int off = kRecentreLanes / 2; off > 0; off >>= 1) out |= __shfl_xor(out, off);
        }
    }
    if (g == 0) {
        PointBox b;
        for (int a = 0; a < 3; a++) {
            b.lo[a] = v[a] - fabsf(v[a]) * 2.384185791015625e-07f;  // 2^-22
            b.hi[a] = -(v[3 + a] - fabsf(v[3 + a]) * 2.384185791015625e-07f);
        }
        b.bad = last > first && (out || !(amax[u] < 1e30f)) ? 1u : 0u;
        b.pad = 0;
        pbox[u] = b;
    }
}

// One level of internal nodes [ls, le), 8 lanes per node, from the deepest level up: the children's boxes
// become the node's record (around the node's centre) and their union its own box.
__global__ __launch_bounds__(256) void k_node_box(const NodeRec *__restrict__ nodes, const uint32_t *__restrict__ child,
                                                 const NodeExt *__restrict__ ext, uint32_t ls, uint32_t le, float scale,
                                                 PointBox *__restrict__ pbox, NodeBox *__restrict__ nbox) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t k = (uint32_t)(t & 7u);
    if (t / 8 >= le - ls) return;
    const uint32_t u = ls + (uint32_t)(t / 8);
    const uint32_t fc = child[u];
    if (fc == 0) return;  // the node's lanes together
    const uint32_t rec = (fc - 1) >> 3, c = (ext[rec].order[k >> 2] >> (8u * (k & 3u))) & 7u;
    const NodeRec nu = nodes[u], nv = nodes[fc + k];
    const PointBox b = pbox[fc + k];
    const bool some = nv.last > nv.first;
    const double d[3] = {nv.cx - nu.cx, nv.cy - nu.cy, nv.cz - nu.cz}, cu[3] = {nu.cx, nu.cy, nu.cz};
    float ch[6] = {}, lo[3], nhi[3], e2 = 0.0f;
    uint32_t bad = some ? b.bad : 0u;
    for (int a = 0; a < 3; a++) {
        lo[a] = nhi[a] = FLT_MAX;
        if (!some) continue;
        const double l = d[a] + (double)b.lo[a], h = d[a] + (double)b.hi[a];
        lo[a] = __double2float_rd(l), nhi[a] = -__double2float_ru(h);
        const float m = (float)(0.5 * (l + h));
        const double half = fmax(h - (double)m, (double)m - l);
        ch[a] = scale * m, ch[3 + a] = scale * __double2float_ru(half * (1.0 + 4.76837158203125e-07));  // 2^-21
        const float e = fabsf(ch[a]) + ch[3 + a];
        e2 += e * e;
        bad |= !(e < 1e15f) ? 1u : 0u;
    }
    uint32_t occ = some ? 1u << c : 0u;
    e2 *= 1.0f + 9.5367431640625e-07f;
    NodeBox *o = nbox + rec;
    ChildBox cb;
    for (int a = 0; a < 3; a++) cb.c[a] = ch[a], cb.h[a] = ch[3 + a];
    cb.n = nv.last - nv.first, cb.gc = child[fc + k];
    cb.ctr[0] = nv.cx, cb.ctr[1] = nv.cy, cb.ctr[2] = nv.cz;
    cb.first = nv.first, cb.amax = ext[rec].amax[c];
    o->ch[c] = cb;
    for (int off = 4; off > 0; off >>= 1) {
        occ |= __shfl_xor(occ, off), bad |= __shfl_xor(bad, off);
        e2 = fmaxf(e2, __shfl_xor(e2, off));
        for (int a = 0; a < 3; a++) lo[a] = fminf(lo[a], __shfl_xor(lo[a], off)), nhi[a] = fminf(nhi[a], __shfl_xor(nhi[a], off));
    }
    if (k < 3) o->c[k] = cu[k];
    if (k == 0) {
        o->ext2 = bad ? __builtin_huge_valf() : e2;
        o->occ = occ;
        PointBox p;
        for (int a = 0; a < 3; a++) p.lo[a] = lo[a], p.hi[a] = -nhi[a];
        p.bad = bad, p.pad = 0;
        pbox[u] = p;
    }
}

hipError_t launch_boxes(oct_ctx *ctx) {
    if (ctx->has_boxes) return hipSuccess;
    const uint32_t nt = ctx->n_total;
    hipError_t e;
    // the nodes' own boxes are needed here only: they lie in the sort's key buffer, which no sort is using
    if ((e = ctx->keys_p.reserve((size_t)nt * (sizeof(PointBox) / sizeof(uint64_t)))) != hipSuccess) return e;
    PointBox *pbox = reinterpret_cast<PointBox *>(ctx->keys_p.p);
    if ((e = ctx->nbox.reserve(ctx->n_internal + 1)) != hipSuccess) return e;
    double ext = 0.0;
    for (int a = 0; a < 3; a++) ext = std::max(ext, 2.0 * fabs(ctx->radii[a]));
    // 2^-k with 2^k in [4, 8] extents; degenerate boxes keep their unit (their squares would leave FP32)
    ctx->box_scale = ext > 1e-15 ? (float)exp2(-ceil(log2(4.0 * ext))) : 1.0f;
    const unsigned nb = (unsigned)(((size_t)nt * kRecentreLanes + 255) / 256);
    LevelTable lt;
    for (uint32_t l = 0; l < kMaxDepth + 3; l++) lt.start[l] = ctx->level_start[l];
    const double mc = std::max(ctx->geo[66], std::max(ctx->geo[67], ctx->geo[68]));
    k_leaf_box<<<nb, 256, 0, ctx->stream>>>(ctx->p64.p, ctx->p32.p, ctx->nodes.p, ctx->child.p, ctx->amax.p, ctx->radtab.p, lt,
                                            mc * 0x1p-49, nt, pbox);
    for (int l = (int)ctx->n_levels - 2; l >= 0; l--) {
        const uint32_t ls = ctx->level_start[l], le = ctx->level_start[l + 1];
        if (le > ls)
            k_node_box<<<(unsigned)(((size_t)(le - ls) * 8 + 255) / 256), 256, 0, ctx->stream>>>(
                ctx->nodes.p, ctx->child.p, ctx->next.p, ls, le, ctx->box_scale, pbox, ctx->nbox.p);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    ctx->has_boxes = true;
    return hipSuccess;
}

template <class T>
static hipError_t grow_preserve(oct_ctx *ctx, DevBuf<T> &b, size_t need, size_t valid) {
    if (need <= b.cap) return hipSuccess;
    size_t cap = b.cap ? b.cap : 1024;
    while (cap < need) cap *= 2;
    T *p = nullptr;
    hipError_t e = hipMalloc((void **)&p, cap * sizeof(T));
    if (e != hipSuccess) return e;
    if (b.p && valid) {
        e = hipMemcpyAsync(p, b.p, valid * sizeof(T), hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) return e;
        e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) return e;
    }
    if (b.p) (void)hipFree(b.p);
    b.p = p;
    b.cap = cap;
    return hipSuccess;
}

hipError_t launch_build(oct_ctx *ctx, uint32_t M, std::string &err) {
    const uint32_t n = (uint32_t)ctx->n;
    BuildGeom g;
    g.encoder = ctx->encoder;
    for (int a = 0; a < 3; a++) g.boxmin[a] = ctx->boxmin[a], g.hl[a] = ctx->half_lengths[a];
    for (int l = 0; l < 22; l++)
        for (int a = 0; a < 3; a++) g.rad[l][a] = ctx->level_radii[l][a];

    hipError_t e;
    // geometry for the searches: level radii, then per axis |centre| + radius (the kNN pruning margin);
    // copied from the context's own array, which outlives the copy
    for (int l = 0; l < 22; l++)
        for (int a = 0; a < 3; a++) ctx->geo[3 * l + a] = ctx->level_radii[l][a];
    for (int a = 0; a < 3; a++) ctx->geo[66 + a] = fabs(ctx->center[a]) + fabs(ctx->radii[a]);
    if ((e = ctx->radtab.reserve(69)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(ctx->radtab.p, ctx->geo, 69 * sizeof(double), hipMemcpyHostToDevice, ctx->stream)) !=
        hipSuccess)
        return e;
    // node capacity: 8 n / M + 64 holds every tree seen (50 M tile, maxLeaf 128: 2.06 M nodes of 3.1 M);
    // the device level loop never grows it, the host loop below does when it must
    const size_t est = 64 + 8 * (size_t)n / (M ? M : 1);
    if ((e = grow_preserve(ctx, ctx->nodes, est, 0)) != hipSuccess) return e;
    if ((e = grow_preserve(ctx, ctx->nkey, est, 0)) != hipSuccess) return e;
    if ((e = grow_preserve(ctx, ctx->child, est + 1, 0)) != hipSuccess) return e;
    if ((e = grow_preserve(ctx, ctx->flags, est, 0)) != hipSuccess) return e;
    if ((e = grow_preserve(ctx, ctx->nrank, est, 0)) != hipSuccess) return e;
    if ((e = ctx->misc.reserve(12 * 1024 + 64)) != hipSuccess) return e;
    uint32_t *total_dev = ctx->misc.p + 8;

    // leaf-recentred FP32 cloud and the children tables, sized for the capacity
    if ((e = ctx->p32.reserve(ctx->n + kPointPad)) != hipSuccess) return e;
    stage_begin(ctx, ST_BUILD);
    const size_t cap = std::min<size_t>(ctx->nodes.cap, ctx->child.cap - 1);
    if (cap < (1ull << 30)) {
        // device level loop, then the recentring and the children tables over the node count the loop
        // leaves on the device: one read-back at the end
        if ((e = ctx->amax.reserve(cap)) != hipSuccess) return e;
        if ((e = ctx->next.reserve((cap + 6) / 8 + 1)) != hipSuccess) return e;
        LevelCtl *ctl = reinterpret_cast<LevelCtl *>(ctx->misc.p + 4096);
        uint32_t *counters = ctx->misc.p + 4096 + 2 * (kLvlCount + 1), *errw = counters + kLvlCount, *totw = errw + 1;
        const size_t maxtiles = std::max<size_t>(kLvlTiles, (cap + kLvlTileMax - 1) / kLvlTileMax), nlook = (size_t)kLvlCount * maxtiles;
        if ((e = ctx->lookback.reserve(nlook + 1)) != hipSuccess) return e;
        const unsigned ig = (unsigned)std::max<size_t>(1, std::min<size_t>((nlook + 255) / 256, 1024));
        k_level_init<<<ig, 256, 0, ctx->stream>>>(ctx->nodes.p, ctx->nkey.p, ctx->flags.p, n, M, g, ctl, ctx->lookback.p, nlook,
                                                  counters, errw, totw);
        int cus = 0;
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device);
        const size_t sgrid = (size_t)std::max(1, cus) * 8;  // resident workgroups
        for (int l = 0; l < (int)kMaxDepth; l++) {
            // level l holds at most min(8^l, cap) nodes: small grids for the top levels
            const size_t nmax = l < 10 ? std::min<size_t>(cap, 1ull << (3 * l)) : cap;
            const uint32_t tn = level_tile(nmax);
            const unsigned gs = (unsigned)std::min(sgrid, (nmax + tn - 1) / tn);
            k_level_step<<<gs, 256, 0, ctx->stream>>>(ctx->sorted_keys, ctx->nodes.p, ctx->nkey.p, ctx->child.p, ctx->flags.p, ctl,
                                                      (uint32_t)l, ctx->lookback.p + (size_t)l * maxtiles, counters + l,
                                                      tn, (uint32_t)cap, M, g, errw, totw);
        }
        k_recentre_dev<<<(unsigned)((cap * kRecentreLanes + 255) / 256), 256, 0, ctx->stream>>>(
            ctx->p64.p, ctx->nodes.p, ctx->child.p, totw, ctx->p32.p, ctx->amax.p);
        k_node_ext_dev<<<(unsigned)((cap * 8 + 255) / 256), 256, 0, ctx->stream>>>(ctx->nodes.p, ctx->nkey.p, ctx->child.p,
                                                                                   ctx->amax.p, totw, ctl, ctx->encoder, ctx->next.p);
        stage_end(ctx, ST_BUILD);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        LevelCtl hc[kLvlCount + 1];
        uint32_t hw[2] = {0, 0};  // error word, node count
        if ((e = hipMemcpyAsync(hc, ctl, sizeof(hc), hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess) return e;
        if ((e = hipMemcpyAsync(hw, errw, sizeof(hw), hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return e;
        if (hw[0] & kLvlErrSpin) {
            err = "build: look-back wait exceeded its bound";
            return hipErrorUnknown;
        }
        // complete within the capacity: done (else the host loop below redoes it)
        if (!(hw[0] & kLvlErrCap) && hw[1] > 0) {
            uint32_t D = 0;  // the deepest non-empty level
            for (int l = 0; l < kLvlCount; l++)
                if (hc[l].le > hc[l].ls) D = (uint32_t)l;
            const uint32_t n_total = hc[D].le;
            if (n_total != hw[1]) {
                err = "build: inconsistent level table";
                return hipErrorUnknown;
            }
            for (uint32_t l = 0; l <= D; l++) ctx->level_start[l] = hc[l].ls;
            for (uint32_t l = D + 1; l < kMaxDepth + 3; l++) ctx->level_start[l] = n_total;
            ctx->n_total = n_total;
            ctx->n_internal = (n_total - 1) / 8;
            ctx->n_leaf = n_total - ctx->n_internal;
            ctx->n_levels = D + 1;
            ctx->max_depth_seen = D;
            ctx->max_points_leaf = M;
            return hipSuccess;
        }
    }

    // host level loop (arrays grown as needed): scan of the split flags, one round trip per level
    uint32_t ls = 0, le = 1, level = 0, n_internal = 0;
    k_root<<<1, 64, 0, ctx->stream>>>(ctx->nodes.p, ctx->nkey.p, ctx->flags.p, n, M, g);
    ctx->level_start[0] = 0;
    ctx->level_start[1] = 1;
    for (;; level++) {
        const uint32_t cnt = le - ls;
        if ((e = exclusive_scan_u32(ctx, ctx->flags.p + ls, ctx->nrank.p + ls, cnt, total_dev)) != hipSuccess) return e;
        uint32_t nint = 0;
        if ((e = hipMemcpyAsync(&nint, total_dev, sizeof(nint), hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return e;
        if (nint > cnt || (nint && level >= kMaxDepth)) {
            err = "build: inconsistent split count";
            return hipErrorUnknown;
        }
        const size_t newle = (size_t)le + 8ull * nint;
        if (newle >= (1ull << 31)) {
            err = "build: node count exceeds 2^31";
            return hipErrorInvalidValue;
        }
        if ((e = grow_preserve(ctx, ctx->nodes, newle, le)) != hipSuccess) return e;
        if ((e = grow_preserve(ctx, ctx->nkey, newle, le)) != hipSuccess) return e;
        if ((e = grow_preserve(ctx, ctx->child, newle + 1, le)) != hipSuccess) return e;
        if ((e = grow_preserve(ctx, ctx->flags, newle, le)) != hipSuccess) return e;
        if ((e = grow_preserve(ctx, ctx->nrank, newle, le)) != hipSuccess) return e;
        unsigned nb = (unsigned)(((size_t)cnt * 8 + 255) / 256);
        k_children<<<nb, 256, 0, ctx->stream>>>(ctx->sorted_keys, ctx->nodes.p, ctx->nkey.p, ctx->child.p, ctx->flags.p + ls,
                                                ctx->nrank.p + ls, ctx->flags.p + le, ls, le, level, M, g);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        n_internal += nint;
        ctx->level_start[level + 2] = (uint32_t)newle;
        if (nint == 0) break;
        ls = le;
        le = (uint32_t)newle;
    }
    const uint32_t n_total = le;
    // sentinel: offsets has nTotal + 1 entries in the reference (linear_octree.hpp:497)
    if ((e = hipMemsetAsync(ctx->child.p + n_total, 0, sizeof(uint32_t), ctx->stream)) != hipSuccess) return e;
    for (uint32_t l = level + 2; l < kMaxDepth + 3; l++) ctx->level_start[l] = n_total;
    ctx->n_total = n_total;
    ctx->n_internal = n_internal;
    ctx->n_leaf = n_total - n_internal;
    ctx->n_levels = level + 1;
    ctx->max_depth_seen = level;
    ctx->max_points_leaf = M;

    if ((e = ctx->amax.reserve(n_total)) != hipSuccess) return e;
    if (n_total) {
        size_t threads = (size_t)n_total * kRecentreLanes;
        unsigned nb = (unsigned)((threads + 255) / 256);
        k_recentre<<<nb, 256, 0, ctx->stream>>>(ctx->p64.p, ctx->nodes.p, ctx->child.p, n_total, ctx->p32.p, ctx->amax.p);
    }
    // children regrouped by corner bits, for the count-mode searches
    if ((e = ctx->next.reserve(n_internal ? n_internal : 1)) != hipSuccess) return e;
    if (n_internal) {
        LevelTable lt;
        for (uint32_t l = 0; l < kMaxDepth + 3; l++) lt.start[l] = ctx->level_start[l];
        unsigned nb = (unsigned)(((size_t)n_total * 8 + 255) / 256);
        k_node_ext<<<nb, 256, 0, ctx->stream>>>(ctx->nodes.p, ctx->nkey.p, ctx->child.p, ctx->amax.p, n_total, ctx->encoder, lt,
                                                ctx->next.p);
    }
    stage_end(ctx, ST_BUILD);
    return hipGetLastError();
}

}  // namespace oct
