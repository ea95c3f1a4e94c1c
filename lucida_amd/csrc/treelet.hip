// Treelet restructuring of the LBVH on the device. No counterpart in the
// reference, whose GPU path traces the LBVH as built (crates/gpu/src/lbvh.rs,
// relayout crates/core/src/lbvh.rs:315-406); the method is Karras and Aila,
// "Fast Parallel Construction of High-Quality Bounding Volume Hierarchies",
// HPG 2013.
//
// After the bit-exact LBVH (Morton sort, Karras hierarchy, fitted boxes), each
// round handles every internal node once its subtrees are final: nodes are
// bucketed by depth and one launch per level, deepest first, handles that
// level. A node of at least LUCIDA_TREELET_MIN_SIZE primitives gets a whole
// wave, which grows a treelet of up to 7 leaves under the node (always
// opening the leaf of largest surface area; the three levels under the
// node are fetched across lanes first), finds the treelet topology of least
// cost by dynamic programming over the 127 leaf subsets (subset boxes and
// counts in LDS, one subset size after another, each subset's partitions
// spread over a group of lanes), and rewrites the treelet's internal nodes in
// place. Smaller nodes only take their cost from their children. A node
// costs CI x area plus its children's costs, or CT x area x primitives as a
// leaf when it holds at most LUCIDA_TREELET_MAX_LEAF; the cheaper one wins,
// the leaf on a tie. The emit pass then lays the tree out as the LBVH's
// relayout does (children adjacent, depth first, left first) with the chosen
// subtrees collapsed into leaves.
//
// The result is deterministic (a node's outcome depends only on its own
// subtree) and equals oracle/treelet.cpp's bit for bit: the same tie-breaks
// and the same float operations, compiled with contraction off.
#include <hip/hip_runtime.h>

#include "context.hpp"

namespace lucida {
namespace {

constexpr uint32_t NONE = 0xFFFFFFFFu;
constexpr int TL_BLOCK = 256;
constexpr int TL_WAVES = TL_BLOCK / 64;
constexpr int LEAVES = LUCIDA_TREELET_LEAVES;
constexpr uint32_t SUBSETS = 1u << LEAVES;
constexpr uint32_t MIN_SIZE = LUCIDA_TREELET_MIN_SIZE;
constexpr uint32_t MAX_LEAF = LUCIDA_TREELET_MAX_LEAF;
constexpr float CI = LUCIDA_TREELET_CI;
constexpr float CT = LUCIDA_TREELET_CT;
constexpr uint32_t LEAF_BIT = 0x100u;  // in a subset's part word: the subset is kept as one leaf
static_assert(LEAVES == 7 && MIN_SIZE >= 3, "one wave covers the 127 subsets of 7 leaves, two per lane");

// One wave's working set for one treelet, by subset of its leaves.
struct TreeletLds {
    float2 cost[SUBSETS];   // least cost; primitives (as bits)
    float box[6][SUBSETS];  // lo xyz, hi xyz
    float area[SUBSETS];
    uint32_t part[SUBSETS];  // left side of the best split | LEAF_BIT
};

// What each lane works on in the dynamic program over the 127 subsets of seven
// leaves. Subsets of m leaves are solved together, 2^LANE_SHIFT[m] lanes to a
// subset (21 x 1, 35 x 1, 35 x 1, 21 x 2, 7 x 8 and 1 x 64 lanes), each taking
// every 2^LANE_SHIFT[m]-th of its 2^(m-1) - 1 partitions. A partition is named by
// its left side, which keeps the subset's lowest leaf; ascending j deposits j's
// bits on the other leaves, so a lane's partitions ascend. Subset 0: idle.
constexpr uint32_t LANE_SHIFT[LEAVES + 1] = {0, 0, 0, 0, 0, 1, 3, 6};
constexpr int lane_parts(int m) { return ((1 << (m - 1)) - 1 + (1 << LANE_SHIFT[m]) - 1) >> LANE_SHIFT[m]; }
constexpr int part_byte(int m) { return m == 2 ? 0 : part_byte(m - 1) + lane_parts(m - 1); }
constexpr int SUBSET_BYTE = part_byte(LEAVES) + lane_parts(LEAVES);  // the lane's subsets of 2, 3, ... leaves
static_assert(SUBSET_BYTE + LEAVES - 1 <= 32, "a lane's program is 32 bytes");
struct alignas(uint4) LaneProgram {  // a lane reads its 32 bytes as two uint4
    uint8_t byte[64][32];
};
static_assert(alignof(LaneProgram) >= alignof(uint4) && sizeof(LaneProgram::byte[0]) % sizeof(uint4) == 0,
              "every lane's row is aligned for its loads");
constexpr int popcount7(int v) { return (v & 1) + (v >> 1 & 1) + (v >> 2 & 1) + (v >> 3 & 1) + (v >> 4 & 1) + (v >> 5 & 1) + (v >> 6 & 1); }
constexpr LaneProgram make_lane_program() {
    LaneProgram t{};
    for (int m = 2; m <= LEAVES; ++m) {
        int group = 0;
        for (int v = 1; v < (int)SUBSETS; ++v) {
            if (popcount7(v) != m) continue;
            const int low = v & -v;
            for (int r = 0; r < 1 << LANE_SHIFT[m]; ++r) {
                const int lane = (group << LANE_SHIFT[m]) + r;
                t.byte[lane][SUBSET_BYTE + m - 2] = (uint8_t)v;
                int at = part_byte(m);
                for (int j = r; j < (1 << (m - 1)) - 1; j += 1 << LANE_SHIFT[m]) {
                    int side = low, rest = v ^ low;
                    for (int b = 1; rest; b <<= 1) {  // j's bits on the other leaves, lowest first
                        const int bit = rest & -rest;
                        if (j & b) side |= bit;
                        rest ^= bit;
                    }
                    t.byte[lane][at++] = (uint8_t)side;
                }
            }
            ++group;
        }
    }
    return t;
}
__constant__ LaneProgram c_program = make_lane_program();

__device__ inline float area(float lx, float ly, float lz, float hx, float hy, float hz) {
    const float dx = hx - lx, dy = hy - ly, dz = hz - lz;
    return 2.0f * (dx * dy + dy * dz + dz * dx);
}

__device__ inline float node_area(const LucidaAabb* box, uint32_t id) {
    const float4* p = reinterpret_cast<const float4*>(box + id);
    const float4 a = p[0], b = p[1];
    return area(a.x, a.y, a.z, b.x, b.y, b.z);
}

// Orders this wave's LDS traffic (the lanes of one wave only).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct TreeArrays {
    uint32_t n, leaf_base;
    uint2* child;       // internal nodes: (left, right)
    uint32_t* parent;   // all nodes
    LucidaAabb* box;    // all nodes
    uint32_t* size;     // internal nodes: primitives below
    float* cost;        // all nodes
    uint32_t* leafy;    // internal nodes: kept as one leaf
    uint32_t* inner;    // internal nodes: internal nodes emitted below (itself included)
};

__device__ inline uint32_t size_of(const TreeArrays& t, uint32_t id) { return id >= t.leaf_base ? 1u : t.size[id]; }
__device__ inline uint32_t inner_of(const TreeArrays& t, uint32_t id) { return id >= t.leaf_base ? 0u : t.inner[id]; }

// A cost with its 4 lowest mantissa bits cleared: monotone in the cost
// (costs are not negative), so comparing keys is a total order.
__device__ inline float cost_key(float c) { return __uint_as_float(__float_as_uint(c) & 0xFFFFFFF0u); }

// Values of one lane in every lane (the lane uniform).
__device__ inline uint32_t lane_u(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lane); }
__device__ inline float lane_f(float v, int lane) { return __uint_as_float(lane_u(__float_as_uint(v), lane)); }

template <int CTRL>
__device__ inline uint32_t dpp_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}

// The best split so far of a subset: least cost key, then least imbalance,
// then least left side.
struct Split {
    float key;
    uint32_t im, side;
    __device__ inline void take(bool valid, float k, uint32_t i, uint32_t s) {
        // no branches: they cost a lone wave more than the comparisons
        const bool better = valid & ((k < key) | ((k == key) & ((i < im) | ((i == im) & (s < side)))));
        key = better ? k : key;
        im = better ? i : im;
        side = better ? s : side;
    }
    template <int CTRL>
    __device__ inline void with_dpp() {
        take(true, __uint_as_float(dpp_u<CTRL>(__float_as_uint(key))), dpp_u<CTRL>(im), dpp_u<CTRL>(side));
    }
};

// The least-cost subtrees over all subsets of M leaves, from the costs of
// their proper subsets (already in LDS). The split chosen is the least (cost,
// imbalance, mask), imbalance being the difference of the two sides' primitive
// counts, with costs compared to 20 mantissa bits (cost_key): among costs
// equal up to their rounding (boxes that coincide, summed in different
// orders) the most even split, so ties do not build chains. A NaN cost is
// never chosen; with every cost NaN the split is the lowest leaf alone.
template <int M>
__device__ inline void solve_size(TreeletLds& L, uint32_t lane, const uint32_t (&prog)[8], uint32_t full) {
    auto byte = [&](int k) { return (prog[k >> 2] >> (8 * (k & 3))) & 0xFFu; };
    constexpr int N = lane_parts(M);
    uint32_t s = byte(SUBSET_BYTE + M - 2);
    if (s > full) s = 0;
    const float inf = __builtin_huge_valf();
    Split best{inf, 0xFFFFFFFFu, 0xFFu};
    const float count_bits = L.cost[s].y;
    const uint32_t count = __float_as_uint(count_bits);
    const float a = L.area[s];
    float2 left[N];
    float right[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {  // side 0 (no partition, or an idle lane): subset 0, not looked at
        const uint32_t side = s ? byte(part_byte(M) + j) : 0u;
        left[j] = L.cost[side];
        right[j] = L.cost[s ^ side].x;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const uint32_t side = s ? byte(part_byte(M) + j) : 0u;
        const float cand = left[j].x + right[j];
        const uint32_t np = __float_as_uint(left[j].y), nq = count - np;
        best.take((side != 0) & (cand == cand), cost_key(cand), np > nq ? np - nq : nq - np, side);
    }
    if (LANE_SHIFT[M] >= 1) best.with_dpp<0xB1>();   // lane ^ 1
    if (LANE_SHIFT[M] >= 2) best.with_dpp<0x4E>();   // lane ^ 2
    if (LANE_SHIFT[M] >= 3) best.with_dpp<0x141>();  // the other half of eight lanes
    if (LANE_SHIFT[M] >= 6) {
        best.with_dpp<0x140>();  // the other half of sixteen
        Split all{lane_f(best.key, 0), lane_u(best.im, 0), lane_u(best.side, 0)};
        for (int row = 16; row < 64; row += 16) all.take(true, lane_f(best.key, row), lane_u(best.im, row), lane_u(best.side, row));
        best = all;
    }
    if (s && (lane & ((1u << LANE_SHIFT[M]) - 1u)) == 0) {
        uint32_t side = best.side;
        float split = inf;
        if (side == 0xFFu)
            side = s & (0u - s);
        else
            split = L.cost[side].x + L.cost[s ^ side].x;
        const float inner = CI * a + split;
        const float leaf = CT * a * (float)count;
        const bool as_leaf = count <= MAX_LEAF && leaf <= inner;
        L.cost[s] = make_float2(as_leaf ? leaf : inner, count_bits);
        L.part[s] = side | (as_leaf ? LEAF_BIT : 0u);
    }
}

// The whole wave rebuilds the treelet under node x (uniform).
//
// What bounds it is the latency of one treelet, as the levels follow each
// other and most hold fewer treelets than the device has wave slots: dependent
// loads, then chains of cross-lane and LDS steps. So every node the treelet may
// take is fetched with all its data in one round of loads, values travel
// between lanes through readlane and DPP rather than LDS, a lane's partitions
// come from a table and are all read before any is compared, and the rebuilt
// nodes are written by a lane each. A level of few treelets takes 14 us (19
// with LDS permutes, bit deposits and one lane rebuilding), the largest of the
// 328,704-triangle mesh (14,880 treelets) 53 us, where the instructions
// themselves bound it; three rounds there 2,655 -> 1,640 us. One workgroup
// walking the top levels without launches took as long a level, 13 us.
__device__ void restructure(const TreeArrays& t, TreeletLds& L, uint32_t lane, uint32_t x) {
    uint32_t prog[8];
    {
        const uint4* q = reinterpret_cast<const uint4*>(c_program.byte[lane]);
        const uint4 a = q[0], b = q[1];
        prog[0] = a.x; prog[1] = a.y; prog[2] = a.z; prog[3] = a.w;
        prog[4] = b.x; prog[5] = b.y; prog[6] = b.z; prog[7] = b.w;
    }
    // The three levels under x, fetched across lanes first: heap slot p < 14
    // (lane p) holds a node; slots 0 and 1 are x's children and slot p >= 2 is
    // child p & 1 of slot (p - 2) / 2. Slots 14 on are taken in pairs for the
    // children of deeper nodes.
    const uint2 c0 = t.child[x];
    uint32_t hid = lane == 0 ? c0.x : (lane == 1 ? c0.y : NONE);
    for (uint32_t lo = 2, hi = 6; lo < 14; lo = hi, hi = 2 * hi + 2) {
        const uint32_t par = __shfl(hid, lane >= 2 ? (lane - 2) >> 1 : 0u, 64);
        if (lane >= lo && lane < hi && par < t.leaf_base) {
            const uint2 c = t.child[par];
            hid = (lane & 1u) ? c.y : c.x;
        }
    }
    // A slot's node: its box, cost, size and emitted-internal count; the area is
    // -1 for a primitive, which is never opened.
    float4 blo = make_float4(0.0f, 0.0f, 0.0f, 0.0f), bhi = blo;
    float harea = -1.0f, hcost = 0.0f;
    uint32_t hsize = 0, hinner = 0;
    auto fetch = [&]() {
        const float4* p = reinterpret_cast<const float4*>(t.box + hid);
        blo = p[0];
        bhi = p[1];
        hcost = t.cost[hid];
        hsize = size_of(t, hid);
        hinner = inner_of(t, hid);
        harea = hid < t.leaf_base ? area(blo.x, blo.y, blo.z, bhi.x, bhi.y, bhi.z) : -1.0f;
    };
    if (hid != NONE) fetch();
    // Grow: lane i < k holds leaf i's slot, area and primitives (0 for one
    // that is a primitive itself); the leaf of largest area, then most
    // primitives (the first such), is replaced by its left child and its
    // right child appended.
    uint32_t slot = lane < 2 ? lane : 0u;
    float leaf_area = lane < 2 ? harea : -1.0f;
    uint32_t leaf_size = lane < 2 && hid < t.leaf_base ? hsize : 0u;
    uint32_t inner_id = lane == 0 ? x : NONE;
    int k = 2, used = 14;
    while (k < LEAVES) {
        int best = -1;
        float best_a = -1.0f;
        uint32_t best_n = 0;
        for (int i = 0; i < k; ++i) {
            const float a = lane_f(leaf_area, i);
            const uint32_t sz = lane_u(leaf_size, i);
            const bool better = (a >= 0.0f) & ((a > best_a) | ((a == best_a) & (sz > best_n)));
            best_a = better ? a : best_a;
            best_n = better ? sz : best_n;
            best = better ? i : best;
        }
        best = __builtin_amdgcn_readfirstlane(best);
        if (best < 0) break;
        const int ep = (int)lane_u(slot, best);
        const uint32_t e = lane_u(hid, ep);
        int px;
        if (ep < 6) {  // its children are in the heap
            px = 2 * ep + 2;
        } else {
            px = used;
            used += 2;
            if ((int)lane == px || (int)lane == px + 1) {
                const uint2 ce = t.child[e];
                hid = (int)lane == px ? ce.x : ce.y;
                fetch();
            }
        }
        const uint32_t cx = lane_u(hid, px), cy = lane_u(hid, px + 1);
        const float ax = lane_f(harea, px), ay = lane_f(harea, px + 1);
        const uint32_t nx = cx < t.leaf_base ? lane_u(hsize, px) : 0u, ny = cy < t.leaf_base ? lane_u(hsize, px + 1) : 0u;
        if (lane == (uint32_t)(k - 1)) inner_id = e;
        if (lane == (uint32_t)best) {
            slot = (uint32_t)px;
            leaf_area = ax;
            leaf_size = nx;
        }
        if (lane == (uint32_t)k) {
            slot = (uint32_t)px + 1;
            leaf_area = ay;
            leaf_size = ny;
        }
        ++k;
    }
    // Subset boxes and counts: lane l covers subsets l + 1 and l + 65; each
    // box is the union of its leaves in ascending leaf order (l + 65 has those
    // of l + 1, then leaf 6).
    const uint32_t full = (1u << k) - 1;
    const uint32_t s0 = lane + 1, s1 = lane + 65;
    const float inf = __builtin_huge_valf();
    float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf}, lo1[3], hi1[3];
    uint32_t n0 = 0, n1 = 0;
    uint32_t leaf_id = NONE, leaf_inner = 0;  // leaf `lane`'s
    float my_cost = 0.0f;
    for (int i = 0; i < k; ++i) {
        const int sl = (int)lane_u(slot, i);
        const bool in0 = s0 >> i & 1u;
        const float ql[3] = {lane_f(blo.x, sl), lane_f(blo.y, sl), lane_f(blo.z, sl)};
        const float qh[3] = {lane_f(bhi.x, sl), lane_f(bhi.y, sl), lane_f(bhi.z, sl)};
        const uint32_t qs = lane_u(hsize, sl);
        if (i == LEAVES - 1) {
            for (int j = 0; j < 3; ++j) {
                lo1[j] = fminf(lo[j], ql[j]);
                hi1[j] = fmaxf(hi[j], qh[j]);
            }
            n1 = n0 + qs;
        }
        for (int j = 0; j < 3; ++j) {
            lo[j] = fminf(lo[j], in0 ? ql[j] : inf);
            hi[j] = fmaxf(hi[j], in0 ? qh[j] : -inf);
        }
        n0 += in0 ? qs : 0u;
        if ((int)lane == i) {
            leaf_id = lane_u(hid, sl);
            leaf_inner = lane_u(hinner, sl);
        }
        const float qc = lane_f(hcost, sl);
        if (s0 == 1u << i) my_cost = qc;
    }
    wave_sync();  // the previous treelet's LDS reads are done
    if (s0 <= full) {
        for (int j = 0; j < 3; ++j) {
            L.box[j][s0] = lo[j];
            L.box[j + 3][s0] = hi[j];
        }
        L.area[s0] = area(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2]);
        L.cost[s0] = make_float2(my_cost, __uint_as_float(n0));
    }
    if (s1 <= full) {
        for (int j = 0; j < 3; ++j) {
            L.box[j][s1] = lo1[j];
            L.box[j + 3][s1] = hi1[j];
        }
        L.area[s1] = area(lo1[0], lo1[1], lo1[2], hi1[0], hi1[1], hi1[2]);
        L.cost[s1] = make_float2(0.0f, __uint_as_float(n1));
    }
    wave_sync();
    // Least costs, subsets of 2 leaves first, then 3, ...
    solve_size<2>(L, lane, prog, full);
    wave_sync();
    if (k >= 3) solve_size<3>(L, lane, prog, full);
    wave_sync();
    if (k >= 4) solve_size<4>(L, lane, prog, full);
    wave_sync();
    if (k >= 5) solve_size<5>(L, lane, prog, full);
    wave_sync();
    if (k >= 6) solve_size<6>(L, lane, prog, full);
    wave_sync();
    if (k >= 7) solve_size<7>(L, lane, prog, full);
    wave_sync();
    // Rebuild in pre-order, left side first, reusing the treelet's internal
    // nodes in the order they were taken: lane j gets the j-th node's subset,
    // id, split and children; the stack of subtrees to come is in lanes too.
    uint32_t st_set = full, st_id = x;  // stack entry `lane`
    uint32_t my_set = 0, my_id = 0, my_part = 0, my_l = 0, my_r = 0;
    int sp = 1, next = 1, nodes = 0;
    while (sp) {
        --sp;
        const uint32_t s = lane_u(st_set, sp), id = lane_u(st_id, sp);
        const uint32_t pw = (uint32_t)__builtin_amdgcn_readfirstlane((int)L.part[s]);
        const uint32_t pm = pw & (SUBSETS - 1), qm = s ^ pm;
        const bool lone = __popc(pm) == 1, rone = __popc(qm) == 1;
        const uint32_t lc = lone ? lane_u(leaf_id, __ffs(pm) - 1) : lane_u(inner_id, next);
        next += lone ? 0 : 1;
        const uint32_t rc = rone ? lane_u(leaf_id, __ffs(qm) - 1) : lane_u(inner_id, next);
        next += rone ? 0 : 1;
        if ((int)lane == nodes) {
            my_set = s;
            my_id = id;
            my_part = pw;
            my_l = lc;
            my_r = rc;
        }
        ++nodes;
        if (!rone) {
            if ((int)lane == sp) {
                st_set = qm;
                st_id = rc;
            }
            ++sp;
        }
        if (!lone) {
            if ((int)lane == sp) {
                st_set = pm;
                st_id = lc;
            }
            ++sp;
        }
    }
    // emitted-internal counts, children (later in pre-order) first
    uint32_t my_inner = 0;
    for (int j = nodes - 1; j >= 0; --j) {
        const uint32_t s = lane_u(my_set, j), pw = lane_u(my_part, j);
        const uint32_t pm = pw & (SUBSETS - 1);
        auto emitted = [&](uint32_t set) {
            if (__popc(set) == 1) return lane_u(leaf_inner, __ffs(set) - 1);
            return lane_u(my_inner, __ffsll((unsigned long long)__ballot(my_set == set)) - 1);
        };
        const uint32_t both = 1u + emitted(pm) + emitted(s ^ pm);
        if ((int)lane == j) my_inner = (pw & LEAF_BIT) ? 0u : both;
    }
    if ((int)lane < nodes) {
        t.child[my_id] = make_uint2(my_l, my_r);
        t.parent[my_l] = my_id;
        t.parent[my_r] = my_id;
        float4* bp = reinterpret_cast<float4*>(t.box + my_id);
        bp[0] = make_float4(L.box[0][my_set], L.box[1][my_set], L.box[2][my_set], 0.0f);
        bp[1] = make_float4(L.box[3][my_set], L.box[4][my_set], L.box[5][my_set], 0.0f);
        const float2 c = L.cost[my_set];
        t.size[my_id] = __float_as_uint(c.y);
        t.cost[my_id] = c.x;
        t.leafy[my_id] = (my_part & LEAF_BIT) ? 1u : 0u;
        t.inner[my_id] = my_inner;
    }
}

// Longest walk to the root a valid tree allows (its depth is far below this);
// a longer one means broken parent links, and the pass stops and reports it.
constexpr uint32_t MAX_CLIMB = 1u << 16;
constexpr uint32_t MAX_LEVELS = 128;  // depth limit of the level schedule

// One node's cost, leaf choice and emitted-internal count from its children's.
__device__ inline void combine(const TreeArrays& t, uint32_t x) {
    const uint2 c = t.child[x];
    const float a = node_area(t.box, x);
    const float split = t.cost[c.x] + t.cost[c.y];
    const float inner = CI * a + split;
    const uint32_t sz = t.size[x];
    const float leaf = CT * a * (float)sz;
    const bool as_leaf = sz <= MAX_LEAF && leaf <= inner;
    t.cost[x] = as_leaf ? leaf : inner;
    t.leafy[x] = as_leaf ? 1u : 0u;
    t.inner[x] = as_leaf ? 0u : 1u + inner_of(t, c.x) + inner_of(t, c.y);
}

// A round is scheduled by depth: every internal node's depth (its walk to the
// root) and class (treelet root or not) are counted per level, the nodes are
// bucketed into per-level lists, and one launch per level, deepest first,
// handles that level's nodes. A node's descendants are all deeper, so they
// are final when it is handled, and rebuilding a treelet touches only nodes
// below its root; launch boundaries order the levels, so no cross-wave
// synchronisation is needed inside a launch.
__global__ __launch_bounds__(256) void k_tl_depth(TreeArrays t, uint32_t* __restrict__ depth,
                                                  uint32_t* __restrict__ level_count, uint32_t* __restrict__ fault) {
    __shared__ uint32_t h[2 * MAX_LEVELS];
    for (int i = threadIdx.x; i < 2 * (int)MAX_LEVELS; i += 256) h[i] = 0;
    __syncthreads();
    const uint32_t x = blockIdx.x * 256 + threadIdx.x;
    if (x < t.n - 1) {
        uint32_t d = 0, cur = x;
        while (cur != 0 && d < MAX_LEVELS) {
            cur = t.parent[cur];
            ++d;
        }
        if (d >= MAX_LEVELS) {
            atomicOr(fault, 8u);
            d = MAX_LEVELS - 1;
        }
        const uint32_t key = 2 * d + (t.size[x] >= MIN_SIZE ? 1u : 0u);
        depth[x] = key;
        atomicAdd(&h[key], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * (int)MAX_LEVELS; i += 256)
        if (h[i]) atomicAdd(&level_count[i], h[i]);
}

// Scatters node ids into the per-(level, class) lists; cursor[key] starts at
// that list's offset.
__global__ __launch_bounds__(256) void k_tl_bucket(uint32_t internal, const uint32_t* __restrict__ depth,
                                                   uint32_t* __restrict__ cursor, uint32_t* __restrict__ list) {
    __shared__ uint32_t h[2 * MAX_LEVELS], base[2 * MAX_LEVELS];
    for (int i = threadIdx.x; i < 2 * (int)MAX_LEVELS; i += 256) h[i] = 0;
    __syncthreads();
    const uint32_t x = blockIdx.x * 256 + threadIdx.x;
    uint32_t key = 0, local = 0;
    if (x < internal) {
        key = depth[x];
        local = atomicAdd(&h[key], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * (int)MAX_LEVELS; i += 256) base[i] = h[i] ? atomicAdd(&cursor[i], h[i]) : 0u;
    __syncthreads();
    if (x < internal) list[base[key] + local] = x;
}

// One level: the first `waves` waves each rebuild the treelet of one node of
// `big` (nodes of at least MIN_SIZE primitives); the lanes of the remaining
// waves each combine one node of `small`.
__global__ __launch_bounds__(TL_BLOCK) void k_tl_level(TreeArrays t, const uint32_t* __restrict__ big,
                                                       uint32_t waves, const uint32_t* __restrict__ small,
                                                       uint32_t count) {
    __shared__ TreeletLds lds[TL_WAVES];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    const uint32_t w = blockIdx.x * TL_WAVES + wave;
    if (w < waves) {
        restructure(t, lds[wave], lane, (uint32_t)__builtin_amdgcn_readfirstlane((int)big[w]));
        return;
    }
    const uint32_t i = (w - waves) * 64 + lane;
    if (i < count) combine(t, small[i]);
}

__global__ __launch_bounds__(256) void k_tl_leaf_cost(TreeArrays t) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k < t.n) t.cost[t.leaf_base + k] = CT * node_area(t.box, t.leaf_base + k);
}

__global__ __launch_bounds__(256) void k_clear_words(uint32_t* __restrict__ p, uint32_t count) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < count) p[i] = 0u;
}

// Bucket cursors: the exclusive prefix sum of the per-(level, class) counts,
// one thread a count; the counts, then the fault word, also to pinned host
// memory, so that the host plans the round's launches while the nodes are
// bucketed.
__global__ __launch_bounds__(2 * MAX_LEVELS) void k_tl_offsets(const uint32_t* __restrict__ count,
                                                               const uint32_t* __restrict__ fault,
                                                               uint32_t* __restrict__ cursor,
                                                               uint32_t* __restrict__ host) {
    __shared__ uint32_t sum[2 * MAX_LEVELS];
    const uint32_t k = threadIdx.x, own = count[k];
    sum[k] = own;
    __syncthreads();
    for (uint32_t o = 1; o < 2 * MAX_LEVELS; o <<= 1) {
        const uint32_t before = k >= o ? sum[k - o] : 0u;
        __syncthreads();
        sum[k] += before;
        __syncthreads();
    }
    cursor[k] = sum[k] - own;
    host[k] = own;
    if (k == 0) host[2 * MAX_LEVELS] = *fault;
}

// Layout: an emitted internal node of pre-order rank R among emitted internal
// nodes has its children at 1 + 2R and 2 + 2R. Each node finds its rank, its
// parent's rank and its first primitive by walking to the root: R counts each
// ancestor plus the emitted internal nodes of every left sibling subtree on
// the way; the first primitive counts the primitives of those left siblings.
// A node under a collapsed ancestor is not emitted, but a primitive still
// takes its place in the leaf order.
__global__ __launch_bounds__(256) void k_treelet_emit(TreeArrays t, const uint32_t* __restrict__ sorted,
                                                      GpuBvhNode* __restrict__ out, uint32_t* __restrict__ order,
                                                      uint32_t* __restrict__ fault) {
    const uint32_t y = blockIdx.x * 256 + threadIdx.x;
    if (y >= 2 * t.n - 1) return;
    bool emitted = true, right = false;
    uint32_t rank = 0, first = 0, sibling_inner = 0, cur = y, steps = 0;
    while (cur != 0) {
        if (++steps == MAX_CLIMB) {
            atomicOr(fault, 2u);
            return;
        }
        const uint32_t p = t.parent[cur];
        const uint2 c = t.child[p];
        if (t.leafy[p]) emitted = false;
        const bool r = c.y == cur;
        const uint32_t li = r ? inner_of(t, c.x) : 0u;
        if (cur == y) {
            right = r;
            sibling_inner = li;
        }
        rank += 1 + li;
        if (r) first += size_of(t, c.x);
        cur = p;
    }
    if (y >= t.leaf_base) {
        if (first >= t.n) {
            atomicOr(fault, 4u);
            return;
        }
        order[first] = sorted[y - t.leaf_base];
    }
    if (!emitted) return;
    const uint32_t slot = y == 0 ? 0u : 1u + 2u * (rank - 1u - sibling_inner) + (right ? 1u : 0u);
    if (slot >= 2 * t.n - 1) {
        atomicOr(fault, 4u);
        return;
    }
    const float4* bp = reinterpret_cast<const float4*>(t.box + y);
    const float4 a = bp[0], b = bp[1];
    GpuBvhNode nd;
    nd.bounds_min[0] = a.x; nd.bounds_min[1] = a.y; nd.bounds_min[2] = a.z;
    nd.bounds_max[0] = b.x; nd.bounds_max[1] = b.y; nd.bounds_max[2] = b.z;
    if (y >= t.leaf_base || t.leafy[y]) {
        nd.left_first = first;
        nd.count = size_of(t, y);
    } else {
        nd.left_first = 1u + 2u * rank;
        nd.count = 0;
    }
    out[slot] = nd;
}

__global__ __launch_bounds__(256) void k_treelet_gather(const GpuTriangle* __restrict__ tris,
                                                        const uint32_t* __restrict__ order, uint32_t n,
                                                        GpuTriangle* __restrict__ out) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k < n) out[k] = tris[order[k]];
}

inline uint32_t blocks_for(size_t n, int block) { return (uint32_t)((n + block - 1) / block); }

}  // namespace

lucida_status bvh_build_treelet_device(lucida_ctx* ctx, const GpuTriangle* tris, size_t n, const float* positions,
                                       uint32_t rounds, GpuBvhNode* nodes, size_t* num_nodes,
                                       uint32_t* prim_indices, GpuTriangle* tris_sorted, float* stage_us) {
    if (stage_us) stage_us[0] = stage_us[1] = stage_us[2] = 0.0f;
    if (rounds > LUCIDA_TREELET_MAX_ROUNDS)
        return set_error(LUCIDA_INVALID_ARG, "treelet BVH: more than LUCIDA_TREELET_MAX_ROUNDS (64) rounds");
    if (n < 2)  // nothing to restructure: the LBVH's single leaf
        return lbvh_build_device(ctx, tris, n, positions, nodes, num_nodes, prim_indices, tris_sorted, nullptr);
    if (n > (1u << 30)) return set_error(LUCIDA_INVALID_ARG, "treelet BVH: more than 2^30 triangles");
    hipStream_t s = ctx->stream;
    StageEvents<4> ev;
    if (stage_us) {
        LUCIDA_HIP(ev.create(), LUCIDA_VALIDATION);
        LUCIDA_HIP(hipEventRecord(ev[0], s), LUCIDA_VALIDATION);
    }
    lucida_status st = lbvh_fit_device(ctx, tris, n, positions);
    if (st != LUCIDA_OK) return st;
    if (stage_us) LUCIDA_HIP(hipEventRecord(ev[1], s), LUCIDA_VALIDATION);
    const size_t internal = n - 1;
    LUCIDA_HIP(ctx->tl_cost.ensure((2 * n - 1) * 4), LUCIDA_OOM);
    LUCIDA_HIP(ctx->tl_leafy.ensure((internal + 1) * 4), LUCIDA_OOM);  // + the fault word
    LUCIDA_HIP(ctx->tl_order.ensure(n * 4), LUCIDA_OOM);
    TreeArrays t;
    t.n = (uint32_t)n;
    t.leaf_base = (uint32_t)internal;
    t.child = ctx->lb_karras.as<uint2>();
    t.parent = ctx->lb_parent.as<uint32_t>();
    t.box = ctx->lb_nodebox.as<LucidaAabb>();
    t.size = ctx->lb_subtree.as<uint32_t>();
    t.inner = t.size + internal;
    t.cost = ctx->tl_cost.as<float>();
    t.leafy = ctx->tl_leafy.as<uint32_t>();
    uint32_t* fault = t.leafy + internal;
    LUCIDA_HIP(ctx->tl_list.ensure((internal + 4 * MAX_LEVELS) * 4), LUCIDA_OOM);
    uint32_t* list = ctx->tl_list.as<uint32_t>();
    uint32_t* level_count = list + internal;
    uint32_t* cursor = level_count + 2 * MAX_LEVELS;
    uint32_t* key = ctx->lb_flags.as<uint32_t>();  // per internal node: 2 x depth + treelet root
    if (!ctx->tl_host)
        LUCIDA_HIP(hipHostMalloc(reinterpret_cast<void**>(&ctx->tl_host), (2 * MAX_LEVELS + 1) * 4,
                                 hipHostMallocDefault),
                   LUCIDA_OOM);
    if (!ctx->tl_counted)
        LUCIDA_HIP(hipEventCreateWithFlags(&ctx->tl_counted, hipEventDisableTiming), LUCIDA_VALIDATION);
    const volatile uint32_t* pinned = ctx->tl_host;
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(256), 0, s, fault, 1u);
    hipLaunchKernelGGL(k_tl_leaf_cost, dim3(blocks_for(n, 256)), dim3(256), 0, s, t);
    for (uint32_t r = 0; r < (rounds ? rounds : 1u); ++r) {
        hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(256), 0, s, level_count, 2 * MAX_LEVELS);
        hipLaunchKernelGGL(k_tl_depth, dim3(blocks_for(internal, 256)), dim3(256), 0, s, t, key, level_count, fault);
        hipLaunchKernelGGL(k_tl_offsets, dim3(1), dim3(2 * MAX_LEVELS), 0, s, level_count, fault, cursor,
                           ctx->tl_host);
        LUCIDA_HIP(hipEventRecord(ctx->tl_counted, s), LUCIDA_VALIDATION);
        hipLaunchKernelGGL(k_tl_bucket, dim3(blocks_for(internal, 256)), dim3(256), 0, s, (uint32_t)internal, key,
                           cursor, list);
        LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
        LUCIDA_HIP(hipEventSynchronize(ctx->tl_counted), LUCIDA_VALIDATION);
        uint32_t host[2 * MAX_LEVELS + 1];
        for (uint32_t k = 0; k <= 2 * MAX_LEVELS; ++k) host[k] = pinned[k];
        if (host[2 * MAX_LEVELS]) return set_error(LUCIDA_VALIDATION, "treelet BVH: deeper than 128 levels");
        uint32_t off[2 * MAX_LEVELS], acc = 0;
        int deepest = 0;
        for (uint32_t k = 0; k < 2 * MAX_LEVELS; ++k) {
            off[k] = acc;
            acc += host[k];
            if (host[k]) deepest = (int)(k / 2);
        }
        for (int d = deepest; d >= 0; --d) {
            const uint32_t nsmall = host[2 * d], nbig = host[2 * d + 1];
            if (!nsmall && !nbig) continue;
            const uint32_t waves = nbig + (nsmall + 63) / 64;
            hipLaunchKernelGGL(k_tl_level, dim3(blocks_for(waves, TL_WAVES)), dim3(TL_BLOCK), 0, s, t,
                               list + off[2 * d + 1], nbig, list + off[2 * d], nsmall);
        }
    }
    if (stage_us) LUCIDA_HIP(hipEventRecord(ev[2], s), LUCIDA_VALIDATION);
    uint32_t* order = prim_indices ? prim_indices : ctx->tl_order.as<uint32_t>();
    hipLaunchKernelGGL(k_treelet_emit, dim3(blocks_for(2 * n - 1, 256)), dim3(256), 0, s, t,
                       ctx->lb_vals.as<uint32_t>(), nodes, order, fault);
    if (tris_sorted)
        hipLaunchKernelGGL(k_treelet_gather, dim3(blocks_for(n, 256)), dim3(256), 0, s, tris, order, (uint32_t)n,
                           tris_sorted);
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    if (stage_us) LUCIDA_HIP(hipEventRecord(ev[3], s), LUCIDA_VALIDATION);
    // the root's emitted-internal count (0 when the root is one leaf)
    uint32_t root_inner = 0, faults = 0;
    LUCIDA_HIP(hipMemcpyAsync(&root_inner, t.inner, 4, hipMemcpyDeviceToHost, s), LUCIDA_READBACK);
    LUCIDA_HIP(hipMemcpyAsync(&faults, fault, 4, hipMemcpyDeviceToHost, s), LUCIDA_READBACK);
    LUCIDA_HIP(hipStreamSynchronize(s), LUCIDA_VALIDATION);
    if (faults || root_inner >= n)
        return set_error(LUCIDA_VALIDATION, "treelet BVH: inconsistent tree (parent links or layout)");
    *num_nodes = 1 + 2 * (size_t)root_inner;
    if (stage_us) {
        for (int k = 0; k < 3; ++k) {
            float ms = 0;
            LUCIDA_HIP(hipEventElapsedTime(&ms, ev[k], ev[k + 1]), LUCIDA_VALIDATION);
            stage_us[k] = ms * 1000.0f;
        }
    }
    return LUCIDA_OK;
}

}  // namespace lucida

using namespace lucida;

extern "C" {

lucida_status lucida_bvh_build_treelet(lucida_ctx* ctx, const GpuTriangle* tris, size_t n, const float* positions,
                                       size_t num_positions, uint32_t rounds, GpuBvhNode* nodes_out,
                                       size_t* num_nodes, uint32_t* prim_indices_out) {
    if (!ctx || !num_nodes || (n && (!tris || !positions || !nodes_out || !prim_indices_out)))
        return set_error(LUCIDA_INVALID_ARG, "lucida_bvh_build_treelet: null argument");
    clear_error();
    if (n == 0) {
        *num_nodes = 0;
        return LUCIDA_OK;
    }
    for (size_t i = 0; i < n; ++i)
        if (tris[i].i0 >= num_positions || tris[i].i1 >= num_positions || tris[i].i2 >= num_positions)
            return set_error(LUCIDA_INVALID_ARG, "lucida_bvh_build_treelet: triangle index out of range");
    hipStream_t s = ctx->stream;
    LUCIDA_HIP(ctx->lb_tris.ensure(n * sizeof(GpuTriangle)), LUCIDA_OOM);
    LUCIDA_HIP(ctx->lb_pos.ensure(num_positions * 16), LUCIDA_OOM);
    LUCIDA_HIP(ctx->lb_nodes.ensure((2 * n - 1) * sizeof(GpuBvhNode)), LUCIDA_OOM);
    LUCIDA_HIP(ctx->lb_prims.ensure(n * 4), LUCIDA_OOM);
    LUCIDA_HIP(hipMemcpyAsync(ctx->lb_tris.ptr, tris, n * sizeof(GpuTriangle), hipMemcpyHostToDevice, s),
               LUCIDA_VALIDATION);
    LUCIDA_HIP(hipMemcpyAsync(ctx->lb_pos.ptr, positions, num_positions * 16, hipMemcpyHostToDevice, s),
               LUCIDA_VALIDATION);
    lucida_status st = bvh_build_treelet_device(ctx, ctx->lb_tris.as<GpuTriangle>(), n, ctx->lb_pos.as<float>(),
                                                rounds, ctx->lb_nodes.as<GpuBvhNode>(), num_nodes,
                                                ctx->lb_prims.as<uint32_t>(), nullptr, nullptr);
    if (st != LUCIDA_OK) return st;
    LUCIDA_HIP(hipMemcpyAsync(nodes_out, ctx->lb_nodes.ptr, *num_nodes * sizeof(GpuBvhNode), hipMemcpyDeviceToHost, s),
               LUCIDA_READBACK);
    LUCIDA_HIP(hipMemcpyAsync(prim_indices_out, ctx->lb_prims.ptr, n * 4, hipMemcpyDeviceToHost, s), LUCIDA_READBACK);
    LUCIDA_HIP(hipStreamSynchronize(s), LUCIDA_VALIDATION);
    return LUCIDA_OK;
}

lucida_status lucida_bvh_build_treelet_device(lucida_ctx* ctx, const GpuTriangle* tris, size_t n,
                                              const float* positions, uint32_t rounds, GpuBvhNode* nodes,
                                              size_t* num_nodes, uint32_t* prim_indices, GpuTriangle* tris_sorted,
                                              float* stage_us) {
    if (!ctx || !num_nodes || (n && (!tris || !positions || !nodes)))
        return set_error(LUCIDA_INVALID_ARG, "lucida_bvh_build_treelet_device: null argument");
    clear_error();
    if (n == 0) {
        *num_nodes = 0;
        return LUCIDA_OK;
    }
    return bvh_build_treelet_device(ctx, tris, n, positions, rounds, nodes, num_nodes, prim_indices, tris_sorted,
                                    stage_us);
}

}  // extern "C"
