// build_tree.hpp -- the binary tree of a build and its collapse: bottom-up
// boxes, treelet restructuring, and the 4-wide nodes (gfx950).
//
// Both bottom-up passes (boxes; boxes with treelets) have to visit a node
// after its whole subtree. A pass is cut by primitive counts: the subtrees of
// at most kTierLow primitives are each taken by one workgroup, which holds
// the subtree in LDS and walks its levels with workgroup barriers; then one
// workgroup per subtree of at most kTierHigh primitives visits the nodes
// above those, and one workgroup the rest. A kernel per tier instead of one
// per depth level, and no host read between them.
#pragma once

#include "rtg_device.hpp"

namespace rtg {

// ---------------------------------------------------------------------------
// Boxes
// ---------------------------------------------------------------------------
// min/max of box planes as selects: the first operand wins ties, so that
// +0/-0 resolve the same way on every device.
__device__ inline float mins(float a, float b) { return b < a ? b : a; }
__device__ inline float maxs(float a, float b) { return b > a ? b : a; }
__device__ inline Box box_union(const Box& a, const Box& b) {
    Box r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = mins(a.lo[k], b.lo[k]);
        r.hi[k] = maxs(a.hi[k], b.hi[k]);
    }
    return r;
}
__device__ inline Box box_empty() {
    Box b;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = __builtin_inff();
        b.hi[k] = -__builtin_inff();
    }
    return b;
}

// Order-preserving map of float to uint (for atomic min/max of centres).
__device__ inline uint32_t f2ord(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float ord2f(uint32_t o) { return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o); }

// Surface area of a box (half of it: the build only compares areas).
__device__ inline float box_area(const Box& b) {
    float ex = b.hi[0] - b.lo[0], ey = b.hi[1] - b.lo[1], ez = b.hi[2] - b.lo[2];
    return (ex * ey + ey * ez) + ez * ex;
}

// A node of the binary tree: its children (internal node number, or kLeafBit
// and a position in the sorted order) beside the areas of those that are
// internal, so that opening a child and ranking what it holds takes one load.
struct alignas(16) BinNode {
    uint32_t left, right;
    float area_l, area_r;
};

constexpr uint32_t kTierLow = 256;     // largest subtree a bottom workgroup holds in LDS
constexpr uint32_t kTierHigh = 65536;  // largest subtree of the middle tier

// ---------------------------------------------------------------------------
// Treelet restructuring (Karras & Aila 2013, HPG, "Fast Parallel
// Construction of High-Quality Bounding Volume Hierarchies", section 4) of
// the binary tree, for single-primitive leaves. The treelet of internal node
// r: r's two children, then, while fewer than kTreeletLeaves, the treelet
// leaf with the largest area that is an internal node replaced by its left
// child in place and its right child appended. Its topology becomes the one
// that minimises the summed surface area of its internal nodes (SAH cost with
// fixed leaves), by dynamic programming over subsets of treelet leaves:
// cost(S) = area(S) + min over partitions (P, S\P), P holding S's lowest
// leaf, of cost(P) + cost(S\P); partitions tried in decreasing order of P,
// the first minimum kept. New internal nodes reuse the treelet's numbers:
// r for the whole set, then the expanded nodes in expansion order, handed
// out as subsets are split from a stack (P's subtree first). A node is
// processed after its whole subtree, so the result does not depend on timing.
//
// One treelet takes a group of G lanes: 16 where a level has treelets for
// several groups of every wave, 64 where it has no more treelets than waves
// and the level's time is one treelet's. Lane k holds treelet leaf k while
// the treelet is formed; the subsets' areas are spread over the lanes by
// their high bits; the dynamic programme goes by subset size, the sets of a
// size (or parts of their partitions) side by side in the lanes, its table
// in LDS. One lane for a whole treelet took 85 us of dependent LDS reads,
// whatever a level's size; a group of 16 takes about 5 us, a chain of some
// 750 VALU operations and 30 LDS round trips of one wave: records read ahead
// of the choice between them, minima over lanes by DPP, a lane's sets in
// registers, the new boxes straight from the leaves (1 M triangles 5,880 ->
// 5,720 us).
// ---------------------------------------------------------------------------
constexpr int kTreeletLeaves = 7;
constexpr int kTreeletRounds = 5;  // passes with RTG_BUILD_PREFER_FAST_TRACE

struct alignas(16) TreeletScratch {
    float cost[1 << kTreeletLeaves];
    float4 leaf[kTreeletLeaves][2];  // lo.xyz, hi.x; hi.yz, area, reference
    uint32_t lcount[8], inner[8];
    uint8_t split[1 << kTreeletLeaves];
    float nbox[kTreeletLeaves - 1][6];  // boxes of the new nodes, where their order matters
    uint32_t pad[4];  // groups of a wave start 16 banks apart
};
static_assert(sizeof(TreeletScratch) % 16 == 0, "scratch records stay 16-byte aligned");
static_assert(sizeof(TreeletScratch) / 4 % 32 == 16, "groups of a wave start 16 banks apart");

// The subsets of 7 treelet leaves by size (2 to 7), ascending within a size,
// so that those of the first m leaves come first.
constexpr int kTreeletSets = 120;
struct TreeletSetTable {
    uint8_t s[kTreeletSets];
    constexpr TreeletSetTable() : s() {
        int n = 0;
        for (int size = 2; size <= kTreeletLeaves; ++size)
            for (int v = 1; v < (1 << kTreeletLeaves); ++v) {
                int bits = 0;
                for (int b = 0; b < kTreeletLeaves; ++b) bits += (v >> b) & 1;
                if (bits == size) s[n++] = (uint8_t)v;
            }
    }
};
__device__ constexpr TreeletSetTable kTreeletSetTable;

constexpr uint32_t binom(uint32_t n, uint32_t k) {
    uint64_t r = 1;
    for (uint32_t i = 0; i < k; ++i) r = r * (n - i) / (i + 1);
    return k > n ? 0u : (uint32_t)r;
}
// number of subsets of size m of n <= 7 leaves, for a fixed m
template <int M>
__device__ __forceinline__ uint32_t set_count(int n) {
    constexpr uint64_t packed = ((uint64_t)binom(2, M) << 16) | ((uint64_t)binom(3, M) << 24) |
                                ((uint64_t)binom(4, M) << 32) | ((uint64_t)binom(5, M) << 40) |
                                ((uint64_t)binom(6, M) << 48) | ((uint64_t)binom(7, M) << 56);
    return (uint32_t)(packed >> (8 * n)) & 0xffu;
}
constexpr int set_offset(int m) {
    int o = 0;
    for (int k = 2; k < m; ++k) o += (int)binom(kTreeletLeaves, k);
    return o;
}

template <int Ctrl>
__device__ __forceinline__ uint32_t dpp_max(uint32_t x) {
    const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, Ctrl, 0xf, 0xf, true);
    return max(x, y);
}
// max over the aligned 8 lanes this lane is in
__device__ __forceinline__ uint32_t max8(uint32_t x) {
    x = dpp_max<0xB1>(x);   // quad_perm 1,0,3,2
    x = dpp_max<0x4E>(x);   // quad_perm 2,3,0,1
    return dpp_max<0x141>(x);  // row_half_mirror
}

// The sets a lane works on, a byte each, in the order of treelet_sizes: fixed
// by its place in the group, so read once per kernel.
template <int G>
struct TreeletLane {
    static constexpr int kWords = G == 16 ? 3 : 2;
    uint32_t w[kWords];
    __device__ __forceinline__ uint32_t set(int k) const { return (w[k / 4] >> (8 * (k % 4))) & 0xffu; }
    template <int M, int L, int K>
    __device__ __forceinline__ void fill(int gl) {
        constexpr int kTasks = (int)binom(kTreeletLeaves, M) * L, kIters = (kTasks + G - 1) / G;
#pragma unroll
        for (int it = 0; it < kIters; ++it) {
            const int task = it * G + gl;
            const uint32_t s = kTreeletSetTable.s[set_offset(M) + (task < kTasks ? task : 0) / L];
            w[(K + it) / 4] |= s << (8 * ((K + it) % 4));
        }
    }
    __device__ __forceinline__ void init() {
        const int gl = threadIdx.x & (G - 1);
#pragma unroll
        for (int k = 0; k < kWords; ++k) w[k] = 0;
        if constexpr (G == 16) {
            fill<2, 1, 0>(gl);
            fill<3, 1, 2>(gl);
            fill<4, 1, 5>(gl);
            fill<5, 2, 8>(gl);
            fill<6, 2, 11>(gl);
        } else {
            fill<2, 1, 0>(gl);
            fill<3, 1, 1>(gl);
            fill<4, 1, 2>(gl);
            fill<5, 2, 3>(gl);
            fill<6, 8, 4>(gl);
        }
    }
};

// One step of split_min: the other lane's (cost, split), taken if it is the
// better or, at the same cost, the larger split. Split 0 holds none; a NaN
// (only the first partition's cost can be one here) is taken as it stands.
__device__ __forceinline__ void split_take(float& best, uint32_t& bp, float co, uint32_t po) {
    const bool less = co < best || (co == best && po > bp);
    const bool take = po != 0u && (bp == 0u || co != co || (best == best && less));
    if (take) {
        best = co;
        bp = po;
    }
}
template <int Ctrl>
__device__ __forceinline__ void split_take_dpp(float& best, uint32_t& bp) {
    const float co =
        __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(best), Ctrl, 0xf, 0xf, true));
    const uint32_t po = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bp, Ctrl, 0xf, 0xf, true);
    split_take(best, bp, co, po);
}
// The least cost and its split over the aligned L lanes this lane is in (L =
// 64: in every lane the wave's).
template <int L>
__device__ __forceinline__ void split_min(float& best, uint32_t& bp) {
    if (L >= 2) split_take_dpp<0xB1>(best, bp);    // quad_perm 1,0,3,2
    if (L >= 4) split_take_dpp<0x4E>(best, bp);    // quad_perm 2,3,0,1
    if (L >= 8) split_take_dpp<0x141>(best, bp);   // row_half_mirror
    if (L >= 16) split_take_dpp<0x140>(best, bp);  // row_mirror
    if (L == 64) {
        float c[4];
        uint32_t p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            c[r] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(best), 16 * r));
            p[r] = (uint32_t)__builtin_amdgcn_readlane((int)bp, 16 * r);
        }
        best = c[0];
        bp = p[0];
#pragma unroll
        for (int r = 1; r < 4; ++r) split_take(best, bp, c[r], p[r]);
    }
}

// Costs and splits of the subsets of M treelet leaves. L lanes share a set:
// lane h of them tries the partitions whose top log2(L) free leaves are the
// complement of h's bits, so that ascending h is descending P. K: the lane's
// first set of this size. The sets of a lane are independent, so their table
// reads go out together; lanes without a set read another's and write none.
template <int G, int M, int L, int K>
__device__ __forceinline__ void treelet_size(TreeletScratch* sc, const TreeletLane<G>& lane, int nl, int gl) {
    if (M > nl) return;
    constexpr int kLog = L == 1 ? 0 : L == 2 ? 1 : L == 4 ? 2 : L == 8 ? 3 : L == 16 ? 4 : 6;
    constexpr int kSteps = 1 << (M - 1 - kLog);
    constexpr int kIters = ((int)binom(kTreeletLeaves, M) * L + G - 1) / G;
    const uint32_t ntask = set_count<M>(nl) * L, h = (uint32_t)gl % L;
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const uint32_t S = M == kTreeletLeaves ? (1u << kTreeletLeaves) - 1u : lane.set(K + it);
        const uint32_t low = S & (0u - S);
        uint32_t R = S ^ low, P0 = low;
#pragma unroll
        for (int b = kLog - 1; b >= 0; --b) {
            const uint32_t top = 0x80000000u >> __builtin_clz(R);
            R ^= top;
            if (!((h >> b) & 1u)) P0 |= top;
        }
        // q runs down over the submasks of R; for h = 0 the first one gives
        // P = S, no partition; the first real one starts the minimum
        // whatever its value (a NaN cost stays the minimum)
        const uint32_t first_h = kSteps > 1 ? 0u : 1u;
        constexpr int first_i = kSteps > 1 ? 1 : 0;
        const float area = sc->cost[S];
        float c[kSteps], best = __builtin_inff();
        uint32_t P[kSteps], bp = 0, q = R;
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            P[i] = P0 | q;
            c[i] = sc->cost[P[i]] + sc->cost[S ^ P[i]];
            q = (q - 1u) & R;
        }
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            bool take = c[i] < best;
            if (i == 0) take = take && h != 0u;
            if (i == first_i) take = take || h == first_h;
            if (take) {
                best = c[i];
                bp = P[i];
            }
        }
        split_min<L>(best, bp);
        if (h == 0 && (uint32_t)(it * G + gl) < ntask) {
            sc->cost[S] = area + best;
            sc->split[S] = (uint8_t)bp;
        }
        if (kSteps >= 8) __builtin_amdgcn_sched_barrier(0);
    }
    wave_order();
}

__device__ __forceinline__ void treelet_planes(const TreeletScratch* sc, float pl[kTreeletLeaves][6]) {
#pragma unroll
    for (int k = 0; k < kTreeletLeaves; ++k) {
        const float4 x = sc->leaf[k][0], y = sc->leaf[k][1];
        pl[k][0] = x.x; pl[k][1] = x.y; pl[k][2] = x.z;
        pl[k][3] = x.w; pl[k][4] = y.x; pl[k][5] = y.y;
    }
}

// Restructures the treelet of node r (three or more primitives below it);
// the G lanes of a group call it together. Store: rec(id), box(ref),
// count(ref), put(id, record, box, count).
template <int G, class Store>
__device__ __forceinline__ void treelet_group(Store& S, uint32_t r, TreeletScratch* sc, TreeletLane<G> lane) {
    static_assert(G == 16 || G == 64, "group sizes");
    // opaque here, or everything that follows from the sets alone is kept in
    // registers across treelets (256 of them, and spills)
#pragma unroll
    for (int k = 0; k < TreeletLane<G>::kWords; ++k) asm volatile("" : "+v"(lane.w[k]));
    constexpr int kLowBits = G == 16 ? 3 : 1;  // subset bits a lane goes through by itself
    const int gl = threadIdx.x & (G - 1);
    const int base = (threadIdx.x & 63) & ~(G - 1);
    // formation: lane k < nl holds leaf k and, if it is an internal node, its
    // record, read ahead of the choice that may open it
    uint32_t ref = kEmpty;
    float area = 0.0f;
    BinNode nd = S.rec(r);
    if (gl == 0) ref = nd.left;
    if (gl == 1) ref = nd.right;
    if (gl < 2 && !(ref & kLeafBit)) {
        nd = S.rec(ref);
        area = box_area(S.box(ref));
    }
    if (gl == 0) sc->inner[0] = r;
    int nl = 2;
    while (nl < kTreeletLeaves) {
        const bool internal = gl < nl && !(ref & kLeafBit);
        // largest area, lowest lane; a NaN area wins only in the first
        // internal leaf and never later, as the comparisons in leaf order do
        const uint32_t cand = (uint32_t)(__ballot(internal) >> base) & 0xffu;
        if (cand == 0) break;
        uint32_t key = internal ? f2ord(area + 0.0f) : 0u;
        if (__ballot(area != area) != 0) {
            if (internal && area != area) key = __builtin_ctz(cand) == gl ? 0xffffffffu : 1u;
        }
        const uint32_t top = max8(key);
        const int best = __builtin_ctz((uint32_t)(__ballot(internal && key == top) >> base) & 0xffu);
        uint32_t right;
        float area_r;
        if (G == 64) {
            right = (uint32_t)__builtin_amdgcn_readlane((int)nd.right, best);
            area_r = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(nd.area_r), best));
        } else {
            right = (uint32_t)__shfl((int)nd.right, best, G);
            area_r = __shfl(nd.area_r, best, G);
        }
        if (gl == best) {
            sc->inner[nl - 1] = ref;
            ref = nd.left;
            area = nd.area_l;
        }
        if (gl == nl) {
            ref = right;
            area = area_r;
        }
        if ((gl == best || gl == nl) && !(ref & kLeafBit)) nd = S.rec(ref);
        ++nl;
    }
    // A box plane that is NaN or -0 makes a box depend on the order its
    // leaves are folded in; without one any order gives the same bits.
    bool ordered = false;
    if (gl < nl) {
        const Box b = S.box(ref);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            ordered = ordered || b.lo[a] != b.lo[a] || __float_as_uint(b.lo[a]) == 0x80000000u;
            ordered = ordered || b.hi[a] != b.hi[a] || __float_as_uint(b.hi[a]) == 0x80000000u;
        }
        sc->leaf[gl][0] = make_float4(b.lo[0], b.lo[1], b.lo[2], b.hi[0]);
        sc->leaf[gl][1] = make_float4(b.hi[1], b.hi[2], area, __uint_as_float(ref));
        sc->lcount[gl] = S.count(ref);
    }
    ordered = ((__ballot(ordered) >> base) & 0xffu) != 0;
    wave_order();
    // areas of the subsets: the lane's high bits choose leaves kLowBits..6.
    // fminf/fmaxf fold the same values as the selects of box_union from the
    // empty box (NaN planes skipped); a zero's sign does not change an area.
    {
        float lo[3], hi[3], pl[kTreeletLeaves][6];
        treelet_planes(sc, pl);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = __builtin_inff();
            hi[a] = -__builtin_inff();
        }
#pragma unroll
        for (int k = kLowBits; k < kTreeletLeaves; ++k) {
            if ((gl >> (k - kLowBits)) & 1) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    lo[a] = fminf(lo[a], pl[k][a]);
                    hi[a] = fmaxf(hi[a], pl[k][3 + a]);
                }
            }
        }
#pragma unroll
        for (int low = 0; low < (1 << kLowBits); ++low) {
            float bl[3], bh[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                bl[a] = lo[a];
                bh[a] = hi[a];
#pragma unroll
                for (int k = 0; k < kLowBits; ++k)
                    if ((low >> k) & 1) {
                        bl[a] = fminf(bl[a], pl[k][a]);
                        bh[a] = fmaxf(bh[a], pl[k][3 + a]);
                    }
            }
            const float ex = bh[0] - bl[0], ey = bh[1] - bl[1], ez = bh[2] - bl[2];
            const uint32_t set = ((uint32_t)gl << kLowBits) | (uint32_t)low;
            if (set < (1u << kTreeletLeaves))
                sc->cost[set] = (set & (set - 1u)) == 0u ? 0.0f : (ex * ey + ey * ez) + ez * ex;
        }
    }
    wave_order();
    if constexpr (G == 16) {
        treelet_size<G, 2, 1, 0>(sc, lane, nl, gl);
        treelet_size<G, 3, 1, 2>(sc, lane, nl, gl);
        treelet_size<G, 4, 1, 5>(sc, lane, nl, gl);
        treelet_size<G, 5, 2, 8>(sc, lane, nl, gl);
        treelet_size<G, 6, 2, 11>(sc, lane, nl, gl);
        treelet_size<G, 7, 16, 0>(sc, lane, nl, gl);
    } else {
        treelet_size<G, 2, 1, 0>(sc, lane, nl, gl);
        treelet_size<G, 3, 1, 1>(sc, lane, nl, gl);
        treelet_size<G, 4, 1, 2>(sc, lane, nl, gl);
        treelet_size<G, 5, 2, 3>(sc, lane, nl, gl);
        treelet_size<G, 6, 8, 4>(sc, lane, nl, gl);
        treelet_size<G, 7, 64, 0>(sc, lane, nl, gl);
    }
    // The new internal nodes in the order they come off the stack: lane j
    // walks down the splits to node j. A node j0 over P and Q is followed by
    // P's internal nodes, |P| - 1 of them, then Q's; splitting it hands out
    // the numbers of those of P and Q that are internal, `next` on. Children
    // as codes: 0..6 a treelet leaf, 8 + x internal node number inner[x].
    const bool mine = gl < nl - 1;
    uint32_t set = (1u << nl) - 1u, id = 0, next = 1, c0 = 0, c1 = 0, np = 0;
    {
        int j0 = 0;
        bool walking = mine;
        while (__ballot(walking) != 0) {
            if (walking) {
                const uint32_t P = sc->split[set], Q = set ^ P;
                np = (uint32_t)__popc(P);
                const uint32_t m0 = np > 1u ? 1u : 0u, m1 = (Q & (Q - 1u)) != 0u ? 1u : 0u;
                if (j0 == gl) {
                    c0 = m0 ? 8u + next : (uint32_t)__builtin_ctz(P);
                    c1 = m1 ? 8u + next + m0 : (uint32_t)__builtin_ctz(Q);
                    walking = false;
                } else {
                    const bool in_p = gl < j0 + (int)np;
                    set = in_p ? P : Q;
                    id = in_p ? next : next + m0;
                    next += m0 + m1 + (in_p || np < 2u ? 0u : np - 2u);
                    j0 += in_p ? 1 : (int)np;
                }
            }
        }
    }
    Box b = box_empty();
    if (__ballot(ordered && mine) == 0) {
        float pl[kTreeletLeaves][6];
        treelet_planes(sc, pl);
#pragma unroll
        for (int k = 0; k < kTreeletLeaves; ++k) {
            const bool in = ((set >> k) & 1u) != 0u;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                b.lo[a] = fminf(b.lo[a], in ? pl[k][a] : __builtin_inff());
                b.hi[a] = fmaxf(b.hi[a], in ? pl[k][3 + a] : -__builtin_inff());
            }
        }
    } else {
        // last to first (children come after their parents)
        for (int j = kTreeletLeaves - 2; j >= 0; --j) {
            if (mine && gl == j) {
                Box x, y;
#pragma unroll
                for (int a = 0; a < 6; ++a) {
                    const float u = c0 < 8u ? reinterpret_cast<const float*>(sc->leaf[c0])[a] : sc->nbox[j + 1][a];
                    const float v = c1 < 8u ? reinterpret_cast<const float*>(sc->leaf[c1])[a]
                                            : sc->nbox[j + (int)np][a];
                    (a < 3 ? x.lo[a % 3] : x.hi[a % 3]) = u;
                    (a < 3 ? y.lo[a % 3] : y.hi[a % 3]) = v;
                }
                b = box_union(x, y);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    sc->nbox[j][a] = b.lo[a];
                    sc->nbox[j][3 + a] = b.hi[a];
                }
            }
            wave_order();
        }
    }
    const float my_area = box_area(b);
    const float area_p = __shfl(my_area, (gl + 1) & (G - 1), G), area_q = __shfl(my_area, (gl + (int)np) & (G - 1), G);
    if (mine) {
        uint32_t count = 0;
#pragma unroll
        for (int k = 0; k < kTreeletLeaves; ++k)
            if ((set >> k) & 1u) count += sc->lcount[k];
        const float4 l0 = sc->leaf[c0 & 7u][1], l1 = sc->leaf[c1 & 7u][1];
        BinNode out;
        out.left = c0 < 8u ? __float_as_uint(l0.w) : sc->inner[c0 - 8u];
        out.area_l = c0 < 8u ? l0.z : area_p;
        out.right = c1 < 8u ? __float_as_uint(l1.w) : sc->inner[c1 - 8u];
        out.area_r = c1 < 8u ? l1.z : area_q;
        S.put(sc->inner[id], out, b, count);
    }
    wave_order();
}

// ---------------------------------------------------------------------------
// Bottom tier: one workgroup per subtree of at most kTierLow primitives.
// The subtree's records live in LDS under local numbers, nodes with three or
// more primitives from the front in breadth-first order (their levels in
// `lv`), nodes with two from the back.
// ---------------------------------------------------------------------------
struct LdsTree {
    BinNode rec_[kTierLow];
    Box box_[kTierLow];
    Box leaf_[kTierLow];
    uint32_t gid[kTierLow];       // node number of a local node
    uint32_t leaf_pos[kTierLow];  // sorted position of a local leaf
    uint16_t cnt[kTierLow];       // primitives below a local node
    uint16_t lv[kTierLow + 1];    // first local node of each level
    uint32_t nfront, nback, nleaf, levels;

    __device__ __forceinline__ BinNode rec(uint32_t i) const { return rec_[i]; }
    __device__ __forceinline__ Box box(uint32_t ref) const {
        return (ref & kLeafBit) ? leaf_[ref & 0xffu] : box_[ref];
    }
    __device__ __forceinline__ uint32_t count(uint32_t ref) const { return (ref & kLeafBit) ? 1u : cnt[ref]; }
    __device__ __forceinline__ void put(uint32_t i, const BinNode& nd, const Box& b, uint32_t c) {
        rec_[i] = nd;
        box_[i] = b;
        cnt[i] = (uint16_t)c;
    }
};


// OPT: treelets, `rounds` passes over the same subtree (more than one only
// where the subtree is the whole tree: between passes the nodes above a
// subtree move its nodes); otherwise boxes only.
// THREADS: see launch_pass.
template <bool OPT, int THREADS>
__global__ __launch_bounds__(THREADS, 4) void k_tree_bottom(BinNode* bin, Box* ibox, uint32_t* rcount,
                                                                const Box* lbox, const uint32_t* roots,
                                                                const uint32_t* nroots, int rounds) {
    __shared__ LdsTree T;
    __shared__ TreeletScratch s_sc[OPT ? THREADS / 16 : 1];
    const uint32_t t = threadIdx.x;
    TreeletLane<64> lane64;
    TreeletLane<16> lane16;
    if (OPT) {
        lane64.init();
        lane16.init();
    }
    const uint32_t nr = *nroots;
    for (uint32_t k = blockIdx.x; k < nr; k += gridDim.x) {
        const uint32_t root = roots[k];
        for (int round = 0; round < rounds; ++round) {
            __syncthreads();
            if (t == 0) {
                const uint32_t rc = rcount[root];
                const bool front = rc >= 3;
                T.gid[front ? 0 : kTierLow - 1] = root;
                T.nfront = front ? 1 : 0;
                T.nback = front ? 0 : 1;
                T.nleaf = 0;
                T.lv[0] = 0;
                T.levels = 0;
            }
            __syncthreads();
            // breadth-first: the front nodes of a level hand out local
            // numbers to their children (order within a level is free: no
            // result depends on local numbers)
            uint32_t b = 0, L = 0;
            while (true) {
                const uint32_t e = T.nfront;
                __syncthreads();
                if (b >= e) break;
                for (uint32_t q = b + t; q < e; q += THREADS) {
                    const uint32_t g = T.gid[q];
                    BinNode nd = bin[g];
                    T.cnt[q] = (uint16_t)rcount[g];
                    uint32_t c[2] = {nd.left, nd.right};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        uint32_t local;
                        if (c[h] & kLeafBit) {
                            local = atomicAdd(&T.nleaf, 1u) & 0xffu;
                            T.leaf_pos[local] = c[h] & kFirstMask;
                            local |= kLeafBit;
                        } else if (rcount[c[h]] >= 3) {
                            local = min(atomicAdd(&T.nfront, 1u), kTierLow - 1);
                            T.gid[local] = c[h];
                        } else {
                            local = (kTierLow - 1 - atomicAdd(&T.nback, 1u)) & 0xffu;
                            T.gid[local] = c[h];
                        }
                        c[h] = local;
                    }
                    nd.left = c[0];
                    nd.right = c[1];
                    T.rec_[q] = nd;
                }
                __syncthreads();
                b = e;
                ++L;
                if (t == 0) T.lv[L] = (uint16_t)e;
                if (L >= kTierLow) break;
            }
            const uint32_t nfront = min(T.nfront, kTierLow), nback = min(T.nback, kTierLow);
            // the two leaves of each back node
            for (uint32_t q = t; q < nback; q += THREADS) {
                const uint32_t i = kTierLow - 1 - q;
                BinNode nd = bin[T.gid[i]];
                const uint32_t l = atomicAdd(&T.nleaf, 2u);
                const uint32_t l0 = l & 0xffu, l1 = (l + 1) & 0xffu;
                T.leaf_pos[l0] = nd.left & kFirstMask;
                T.leaf_pos[l1] = nd.right & kFirstMask;
                const Box b0 = lbox[nd.left & kFirstMask], b1 = lbox[nd.right & kFirstMask];
                T.box_[i] = box_union(b0, b1);
                T.leaf_[l0] = b0;
                T.leaf_[l1] = b1;
                nd.left = kLeafBit | l0;
                nd.right = kLeafBit | l1;
                nd.area_l = nd.area_r = 0.0f;
                T.rec_[i] = nd;
                T.cnt[i] = 2;
            }
            // the leaves of the front nodes
            for (uint32_t q = t; q < nfront; q += THREADS) {
                const BinNode nd = T.rec_[q];
                if (nd.left & kLeafBit) T.leaf_[nd.left & 0xffu] = lbox[T.leaf_pos[nd.left & 0xffu]];
                if (nd.right & kLeafBit) T.leaf_[nd.right & 0xffu] = lbox[T.leaf_pos[nd.right & 0xffu]];
            }
            __syncthreads();
            for (uint32_t lev = L; lev-- > 0;) {
                const uint32_t lb = T.lv[lev], le = T.lv[lev + 1];
                if (!OPT) {
                    for (uint32_t q = lb + t; q < le; q += THREADS) {
                        BinNode nd = T.rec_[q];
                        const Box x = T.box(nd.left), y = T.box(nd.right);
                        T.box_[q] = box_union(x, y);
                        nd.area_l = box_area(x);
                        nd.area_r = box_area(y);
                        T.rec_[q] = nd;
                    }
                } else if (le - lb <= THREADS / 64) {
                    const uint32_t w = t >> 6;
                    if (lb + w < le) treelet_group<64>(T, lb + w, &s_sc[w], lane64);
                } else {
                    for (uint32_t q = lb + (t >> 4); q < le; q += THREADS / 16)
                        treelet_group<16>(T, q, &s_sc[t >> 4], lane16);
                }
                __syncthreads();
            }
            // back to the tree under its own numbers
            for (uint32_t q = t; q < nfront + nback; q += THREADS) {
                const uint32_t i = q < nfront ? q : kTierLow - 1 - (q - nfront);
                BinNode nd = T.rec_[i];
                nd.left = (nd.left & kLeafBit) ? (kLeafBit | T.leaf_pos[nd.left & 0xffu]) : T.gid[nd.left];
                nd.right = (nd.right & kLeafBit) ? (kLeafBit | T.leaf_pos[nd.right & 0xffu]) : T.gid[nd.right];
                const uint32_t g = T.gid[i];
                bin[g] = nd;
                ibox[g] = T.box_[i];
                if (OPT) rcount[g] = T.cnt[i];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Upper tiers: one workgroup per subtree visits its nodes of more than
// `lowest` primitives, from the deepest of their levels up, in the tree's own
// (global) records. `list` and `levels` hold each subtree's nodes breadth
// first and their level starts; a subtree of c primitives takes c entries of
// each (it has fewer nodes), from `bump` on.
// ---------------------------------------------------------------------------
struct GlobalTree {
    BinNode* bin;
    Box* ibox;
    uint32_t* rcount;
    const Box* lbox;
    __device__ __forceinline__ BinNode rec(uint32_t i) const { return bin[i]; }
    __device__ __forceinline__ Box box(uint32_t ref) const {
        return (ref & kLeafBit) ? lbox[ref & kFirstMask] : ibox[ref];
    }
    __device__ __forceinline__ uint32_t count(uint32_t ref) const { return (ref & kLeafBit) ? 1u : rcount[ref]; }
    __device__ __forceinline__ void put(uint32_t i, const BinNode& nd, const Box& b, uint32_t c) {
        bin[i] = nd;
        ibox[i] = b;
        rcount[i] = c;
    }
};

constexpr int kUpperThreads = 512;

template <bool OPT>
__global__ __launch_bounds__(kUpperThreads) void k_tree_upper(GlobalTree T, const uint32_t* roots,
                                                              const uint32_t* nroots, uint32_t lowest, uint32_t n,
                                                              uint32_t* list_all, uint32_t* levels_all,
                                                              uint32_t* bump) {
    __shared__ TreeletScratch s_sc[OPT ? kUpperThreads / 16 : 1];
    __shared__ uint32_t s_count, s_base;
    const uint32_t t = threadIdx.x;
    TreeletLane<64> lane64;
    TreeletLane<16> lane16;
    if (OPT) {
        lane64.init();
        lane16.init();
    }
    const uint32_t nr = *nroots;
    for (uint32_t k = blockIdx.x; k < nr; k += gridDim.x) {
        const uint32_t root = roots[k];
        __syncthreads();
        if (t == 0) {
            s_base = atomicAdd(bump, T.rcount[root]);
            s_count = 1;
        }
        __syncthreads();
        const uint32_t base = s_base;
        if (base >= n) return;  // (never: the subtrees of a tier share no primitive)
        const uint32_t cap = n - base;
        uint32_t* list = list_all + base;
        uint32_t* lv = levels_all + base;
        if (t == 0) {
            list[0] = root;
            lv[0] = 0;
        }
        __syncthreads();
        uint32_t b = 0, L = 0;
        while (true) {
            const uint32_t e = min(s_count, cap);
            __syncthreads();
            if (b >= e) break;
            for (uint32_t q = b + t; q < e; q += kUpperThreads) {
                const BinNode nd = T.bin[list[q]];
                const uint32_t c[2] = {nd.left, nd.right};
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (!(c[h] & kLeafBit) && T.rcount[c[h]] > lowest) {
                        const uint32_t at = atomicAdd(&s_count, 1u);
                        if (at < cap) list[at] = c[h];
                    }
            }
            b = e;
            ++L;
            if (t == 0 && L < cap) lv[L] = e;
            __syncthreads();
        }
        for (uint32_t lev = L; lev-- > 0;) {
            const uint32_t lb = lv[lev], le = lev + 1 < L ? lv[lev + 1] : b;
            if (!OPT) {
                for (uint32_t q = lb + t; q < le; q += kUpperThreads) {
                    const uint32_t g = list[q];
                    BinNode nd = T.bin[g];
                    const Box x = T.box(nd.left), y = T.box(nd.right);
                    T.ibox[g] = box_union(x, y);
                    nd.area_l = box_area(x);
                    nd.area_r = box_area(y);
                    T.bin[g] = nd;
                }
            } else if (le - lb <= kUpperThreads / 64) {
                const uint32_t w = t >> 6;
                if (lb + w < le) treelet_group<64>(T, list[lb + w], &s_sc[w], lane64);
            } else {
                for (uint32_t q = lb + (t >> 4); q < le; q += kUpperThreads / 16)
                    treelet_group<16>(T, list[q], &s_sc[t >> 4], lane16);
            }
            __syncthreads();
        }
    }
}

// Roots of the bottom and middle tiers: internal children of at most
// kTierLow (kTierHigh) primitives under a node of more, handed to
// add(tier, node). Their order is free: a tier's subtrees share no node.
template <class Add>
__device__ inline void tier_roots(uint32_t i, uint32_t count, const uint32_t* child, const uint32_t* child_count,
                                  Add add) {
    if (i == 0) {
        if (count <= kTierLow) add(0, 0u);
        else if (count <= kTierHigh) add(1, 0u);
    }
    if (count <= kTierLow) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (child[h] & kLeafBit) continue;
        if (child_count[h] <= kTierLow) add(0, child[h]);
        else if (count > kTierHigh && child_count[h] <= kTierHigh) add(1, child[h]);
    }
}

// The roots a workgroup of kRootThreads nodes found, collected in LDS so that
// each list costs one global atomic: with one per root, 13 ns each on the
// same address, the 4,800 roots among 1 M primitives took 61 us of a
// k_tier_roots of the same length and most of k_karras's 84 us.
constexpr int kRootThreads = 1024;
struct RootList {
    uint32_t node[2][2 * kRootThreads + 1];
    uint32_t n[2], base[2];
    __device__ inline void clear() {
        if (threadIdx.x < 2) n[threadIdx.x] = 0;
        __syncthreads();
    }
    __device__ inline void add(int tier, uint32_t i) { node[tier][atomicAdd(&n[tier], 1u)] = i; }
    // counts[0], counts[1]: how many roots `low` and `mid` hold
    __device__ inline void write(uint32_t* low, uint32_t* mid, uint32_t* counts) {
        __syncthreads();
        if (threadIdx.x < 2 && n[threadIdx.x]) base[threadIdx.x] = atomicAdd(&counts[threadIdx.x], n[threadIdx.x]);
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < n[0]; k += kRootThreads) low[base[0] + k] = node[0][k];
        for (uint32_t k = threadIdx.x; k < n[1]; k += kRootThreads) mid[base[1] + k] = node[1][k];
    }
};

__global__ __launch_bounds__(kRootThreads) void k_tier_roots(uint32_t n, const BinNode* bin, const uint32_t* rcount,
                                                             uint32_t* low, uint32_t* mid, uint32_t* counts) {
    __shared__ RootList R;
    R.clear();
    const uint32_t i = blockIdx.x * kRootThreads + threadIdx.x;
    const uint32_t c = i < n - 1 ? rcount[i] : 0u;
    if (c > kTierLow || (i == 0 && c > 0)) {
        const BinNode nd = bin[i];
        const uint32_t child[2] = {nd.left, nd.right};
        uint32_t cc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) cc[h] = (child[h] & kLeafBit) ? 1u : rcount[child[h]];
        tier_roots(i, c, child, cc, [&](int tier, uint32_t k) { R.add(tier, k); });
    }
    R.write(low, mid, counts);
}

// ---------------------------------------------------------------------------
// Collapse into 4-wide nodes, breadth first. A wide node's slots: the binary
// root's two children, then the largest-area internal slot replaced in place
// by its two children while fewer than four (first slot on ties). Slot boxes
// are the binary tree's: a fold of box planes in leaf order gives the same
// value however it is grouped, as long as no plane is NaN (k_wide_boxes
// below folds them again where one is).
// ---------------------------------------------------------------------------
struct WideTree {
    const BinNode* bin;
    const Box* ibox;
    const Box* lbox;
    Node* nodes;
    uint32_t* wroot;  // binary root of each wide node
    uint32_t cap;     // node capacity (n - 1: every wide node has two or more slots)
};

// Slots of the wide node rooted at binary node r and how many of them become
// wide nodes.
__device__ inline uint32_t wide_slots(const BinNode* bin, uint32_t r, uint32_t s[4]) {
    BinNode nd = bin[r];
    float a[4] = {nd.area_l, nd.area_r, 0.0f, 0.0f};
    s[0] = nd.left;
    s[1] = nd.right;
    s[2] = s[3] = kEmpty;
#pragma unroll
    for (int nslot = 2; nslot < 4; ++nslot) {
        int best = -1;
        float best_area = 0.0f;
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < nslot; ++k) {
            if (s[k] & kLeafBit) continue;
            if (best < 0 || a[k] > best_area) {
                best = k;
                best_area = a[k];
                c = s[k];
            }
        }
        if (best < 0) break;
        nd = bin[c];
#pragma unroll
        for (int k = 3; k >= 1; --k) {
            if (k > best + 1) {
                s[k] = s[k - 1];
                a[k] = a[k - 1];
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k == best) {
                s[k] = nd.left;
                a[k] = nd.area_l;
            }
            if (k == best + 1) {
                s[k] = nd.right;
                a[k] = nd.area_r;
            }
        }
    }
    uint32_t internal = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) internal += (s[k] & kLeafBit) ? 0u : 1u;  // kEmpty has the leaf bit
    return internal;
}

// Writes wide node w of binary slots s; its internal slots take the node
// numbers from `next` on.
__device__ inline void wide_emit(const WideTree& W, uint32_t w, const uint32_t s[4], uint32_t next) {
    float lo[3][4], hi[3][4];
    uint32_t ref[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        Box b = box_empty();
        uint32_t r = s[k];
        if (r != kEmpty) {
            if (r & kLeafBit) {
                b = box_union(b, W.lbox[r & kFirstMask]);
            } else {
                b = W.ibox[r];
                if (next < W.cap) W.wroot[next] = r;
                r = next++;
            }
        }
        ref[k] = r;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a][k] = b.lo[a];
            hi[a][k] = b.hi[a];
        }
    }
    float4* out = reinterpret_cast<float4*>(W.nodes + w);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        out[2 * a] = make_float4(lo[a][0], lo[a][1], lo[a][2], lo[a][3]);
        out[2 * a + 1] = make_float4(hi[a][0], hi[a][1], hi[a][2], hi[a][3]);
    }
    reinterpret_cast<uint4*>(out)[6] = make_uint4(ref[0], ref[1], ref[2], ref[3]);
    reinterpret_cast<uint4*>(out)[7] = make_uint4(0u, 0u, 0u, 0u);
}

// Inclusive prefix sum over the workgroup (part: one word per wave).
template <int BS>
__device__ inline uint32_t block_scan(uint32_t v, uint32_t* part, uint32_t& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)v, off);
        if (lane >= off) v += u;
    }
    if (lane == 63) part[w] = v;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < BS / 64; ++k) {
        const uint32_t p = part[k];
        if (k < w) before += p;
        all += p;
    }
    total = all;
    __syncthreads();
    return v + before;
}

// Progress of a collapse: level L holds nodes [off[L], off[L + 1]); `level`
// is the first level not emitted.
struct CollapseState {
    uint32_t level, nodes, done, pad;
};
// What the host reads after a build's kernels (host memory, written by the device).
constexpr uint32_t kReportLevels = 60;
struct BuildReport {
    uint32_t levels, nodes, done, status, nan_boxes, pad[3];
    uint32_t off[kReportLevels + 1];  // the first level offsets
};

// The first levels, by one workgroup, until one holds more than `most`
// nodes or there is none left.
constexpr int kCollapseThreads = 1024;
__global__ __launch_bounds__(kCollapseThreads) void k_collapse_top(WideTree W, uint32_t most, uint32_t* off,
                                                                   CollapseState* state) {
    __shared__ uint32_t part[kCollapseThreads / 64];
    uint32_t lb = 0, le = 1, level = 0;
    if (threadIdx.x == 0) {
        W.wroot[0] = 0;
        off[0] = 0;
        off[1] = 1;
    }
    __syncthreads();
    while (le - lb <= most && le > lb) {
        uint32_t next = le;
        for (uint32_t q = lb; q < le; q += kCollapseThreads) {
            const uint32_t w = q + threadIdx.x;
            uint32_t s[4], want = 0, total;
            if (w < le) want = wide_slots(W.bin, W.wroot[w], s);
            const uint32_t incl = block_scan<kCollapseThreads>(want, part, total);
            if (w < le) wide_emit(W, w, s, next + incl - want);
            next += total;
        }
        next = min(next, W.cap);
        ++level;
        if (threadIdx.x == 0) off[level + 1] = next;
        lb = le;
        le = next;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        state->level = level;
        state->nodes = le;
        state->done = le == lb ? 1u : 0u;
    }
}

// A later level by many workgroups, 256 nodes a turn: their slots, which
// k_wide_expand found for the first of these levels and the level before for
// the others, give the children's numbers after those of the turns before;
// the nodes are written, and the children's slots with the counts of each
// turn of the next level. `sums`: the turns' counts, three rows of `stride`
// words used in turn (read, filled, cleared). `step`: levels since the one
// that state->level names. One launch a level: with the slots found in a
// launch of their own, 82,000 triangles without treelets took 482 us
// to build and 470 this way.
constexpr uint32_t kWideBlocks = 1024;  // most workgroups of a launch
constexpr uint32_t kWideTurn = 256;

__global__ __launch_bounds__(kWideTurn) void k_wide_expand(WideTree W, const uint32_t* off, const CollapseState* state,
                                                           uint4* slots, uint32_t* sums, uint32_t stride) {
    __shared__ uint32_t part[kWideTurn / 64];
    const uint32_t lb = off[state->level], m = off[state->level + 1] - lb;
    for (uint32_t k = blockIdx.x * kWideTurn + threadIdx.x; k < 2 * stride; k += gridDim.x * kWideTurn)
        sums[stride + k] = 0;
    for (uint32_t c = blockIdx.x; c * kWideTurn < m; c += gridDim.x) {
        const uint32_t q = c * kWideTurn + threadIdx.x;
        uint32_t want = 0, total;
        if (q < m) {
            uint32_t s[4];
            want = wide_slots(W.bin, W.wroot[lb + q], s);
            slots[lb + q] = make_uint4(s[0], s[1], s[2], s[3]);
        }
        block_scan<kWideTurn>(want, part, total);
        if (threadIdx.x == 0) sums[c] = total;
    }
}

__global__ __launch_bounds__(kWideTurn) void k_wide_level(WideTree W, uint32_t* off, const CollapseState* state,
                                                          uint32_t step, uint4* slots, uint32_t* sums,
                                                          uint32_t stride) {
    constexpr uint32_t kSpan = 4 + 2;  // turns of the next level that a turn's children reach into
    __shared__ uint32_t part[kWideTurn / 64], s_next[kSpan];
    const uint32_t L = state->level + step;
    const uint32_t lb = off[L], le = off[L + 1], m = le - lb;
    const uint32_t* cur = sums + (size_t)(step % 3) * stride;
    uint32_t* fill = sums + (size_t)((step + 1) % 3) * stride;
    uint32_t* clear = sums + (size_t)((step + 2) % 3) * stride;
    for (uint32_t k = blockIdx.x * kWideTurn + threadIdx.x; k < stride; k += gridDim.x * kWideTurn) clear[k] = 0;
    if (m == 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) off[L + 2] = le;
        return;
    }
    for (uint32_t c = blockIdx.x; c * kWideTurn < m; c += gridDim.x) {
        uint32_t before = 0, total;
        for (uint32_t k = threadIdx.x; k < c; k += kWideTurn) before += cur[k];
        if (threadIdx.x < kSpan) s_next[threadIdx.x] = 0;
        block_scan<kWideTurn>(before, part, total);
        const uint32_t start = le + total, first = total / kWideTurn, q = c * kWideTurn + threadIdx.x;
        uint32_t s[4] = {kEmpty, kEmpty, kEmpty, kEmpty}, want = 0;
        if (q < m) {
            const uint4 v = slots[lb + q];
            s[0] = v.x;
            s[1] = v.y;
            s[2] = v.z;
            s[3] = v.w;
#pragma unroll
            for (int k = 0; k < 4; ++k) want += (s[k] & kLeafBit) ? 0u : 1u;
        }
        const uint32_t incl = block_scan<kWideTurn>(want, part, total);
        if (q < m) {
            uint32_t at = start + incl - want;
            wide_emit(W, lb + q, s, at);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (s[k] & kLeafBit) continue;
                if (at < W.cap) {
                    uint32_t t[4];
                    const uint32_t n = wide_slots(W.bin, s[k], t);
                    slots[at] = make_uint4(t[0], t[1], t[2], t[3]);
                    if (n) atomicAdd(&s_next[(at - le) / kWideTurn - first], n);
                }
                ++at;
            }
        }
        __syncthreads();
        if (threadIdx.x < kSpan && s_next[threadIdx.x]) atomicAdd(&fill[first + threadIdx.x], s_next[threadIdx.x]);
        if (c == (m - 1) / kWideTurn && threadIdx.x == 0) off[L + 2] = min(start + total, W.cap);
        __syncthreads();
    }
}

// Moves the state past `steps` levels.
__global__ void k_collapse_advance(const uint32_t* off, CollapseState* state, uint32_t steps) {
    if (threadIdx.x != 0) return;
    uint32_t L = state->level;
    for (uint32_t k = 0; k < steps && off[L + 1] > off[L]; ++k) ++L;
    state->level = L;
    state->nodes = off[L + 1];
    state->done = off[L + 1] == off[L] ? 1u : 0u;
}

__global__ __launch_bounds__(64) void k_build_report(const CollapseState* state, const uint32_t* off,
                                                     const uint32_t* status, const uint32_t* nan_boxes,
                                                     BuildReport* out) {
    if (threadIdx.x <= min(state->level, kReportLevels)) out->off[threadIdx.x] = off[threadIdx.x];
    if (threadIdx.x != 0) return;
    out->levels = state->level;
    out->nodes = state->nodes;
    out->done = state->done;
    out->status = *status;
    out->nan_boxes = *nan_boxes;
}

}  // namespace rtg
