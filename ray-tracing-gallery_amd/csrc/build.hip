// build.hip -- acceleration-structure builds on gfx950.
//
// Replaces the driver work behind
//   AccelerationStructure::build_blas   src/util_structs.rs:140-224
//   build_tlas                          src/util_functions.rs:453-510
//   AccelerationStructure::update_tlas  src/util_structs.rs:285-357 (refit)
//   AccelerationStructure::clone        src/util_structs.rs:359-405
// with a linear BVH (Karras 2012): primitive boxes and centres, 30-bit Morton
// codes, a stable LSD radix sort written here (LDS digit ranking with wave
// ballots), the radix-tree split search, bottom-up boxes with the treelet
// passes and a top-down collapse into 4-wide nodes (build_tree.hpp). Up to
// kSmallBuild primitives go from their inputs to the binary tree in one
// workgroup. The blobs are bit-identical to the host oracle's: every box
// operation is an exact min/max or a fixed FP32 sequence.
#include <algorithm>
#include <cstring>
#include <vector>

#include "build_tree.hpp"
#include "rtg_device.hpp"
#include "rtg_internal.hpp"

namespace rtg {

__device__ inline float centre(const Box& b, int a) { return (b.lo[a] + b.hi[a]) * 0.5f + 0.0f; }

__device__ inline void set_slot(Node& nd, int s, const Box& b) {
    nd.lo_x[s] = b.lo[0];
    nd.hi_x[s] = b.hi[0];
    nd.lo_y[s] = b.lo[1];
    nd.hi_y[s] = b.hi[1];
    nd.lo_z[s] = b.lo[2];
    nd.hi_z[s] = b.hi[2];
}

__device__ inline Box slot_box(const Node& nd, int s) {
    Box b;
    b.lo[0] = nd.lo_x[s];
    b.hi[0] = nd.hi_x[s];
    b.lo[1] = nd.lo_y[s];
    b.hi[1] = nd.hi_y[s];
    b.lo[2] = nd.lo_z[s];
    b.hi[2] = nd.hi_z[s];
    return b;
}

// Box of a node: its four slot boxes folded in slot order.
__device__ inline Box node_box(const Node& nd) {
    Box b = box_empty();
#pragma unroll
    for (int s = 0; s < 4; ++s) b = box_union(b, slot_box(nd, s));
    return b;
}

// Slot box of child ref c: its leaf's primitive boxes (leaf_boxes[order[k]],
// or leaf_boxes[k] without an order) folded in leaf order, or its node's box.
__device__ inline Box ref_box(const Node* nodes, uint32_t c, const Box* leaf_boxes, const uint32_t* order) {
    Box b = box_empty();
    if (c == kEmpty) return b;
    if (c & kLeafBit) {
        uint32_t f = c & kFirstMask, cnt = ((c >> 27) & 0xfu) + 1u;
        for (uint32_t k = f; k < f + cnt; ++k) b = box_union(b, leaf_boxes[order ? order[k] : k]);
        return b;
    }
    return node_box(nodes[c]);
}

// Centre bounds of this thread's primitives, folded over the workgroup after.
struct CentreBounds {
    uint32_t lo[3], hi[3];
    __device__ inline CentreBounds() {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = 0xffffffffu;
            hi[a] = 0u;
        }
    }
    __device__ inline void add(const Box& b) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float c = centre(b, a);
            if (!isfinite(c)) continue;
            lo[a] = min(lo[a], f2ord(c));
            hi[a] = max(hi[a], f2ord(c));
        }
    }
};

// Block-wide reduction of centre bounds, then one atomic per block and bound.
template <int BS>
__device__ inline void reduce_centre_bounds(const CentreBounds& c, uint32_t* cb) {
    __shared__ uint32_t s_lo[3][BS / 64], s_hi[3][BS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        uint32_t lo = c.lo[a], hi = c.hi[a];
        for (int off = 32; off > 0; off >>= 1) {
            lo = min(lo, (uint32_t)__shfl_xor((int)lo, off));
            hi = max(hi, (uint32_t)__shfl_xor((int)hi, off));
        }
        if (lane == 0) {
            s_lo[a][w] = lo;
            s_hi[a][w] = hi;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int a = threadIdx.x;
        uint32_t lo = 0xffffffffu, hi = 0u;
        for (int k = 0; k < BS / 64; ++k) {
            lo = min(lo, s_lo[a][k]);
            hi = max(hi, s_hi[a][k]);
        }
        if (lo != 0xffffffffu) atomicMin(&cb[a], lo);
        if (hi != 0u) atomicMax(&cb[3 + a], hi);
    }
}
// k_tri_setup's workgroups, and the most of them: their atomics on the six
// bounds pass one after another (1 M triangles: 99 us with 3,906 workgroups
// of 256 lanes, 33 with these).
constexpr int kSetupThreads = 1024;
constexpr unsigned kSetupBlocks = 512;

struct GeomDesc {
    const uint8_t* vertices;
    const uint32_t* indices;
    uint32_t stride;
    uint32_t max_vertex;
    uint32_t first_tri;
    uint32_t flags;
};

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Words a build clears before its kernels: the centre bounds (cb[0..2] the
// least, cb[3..5] the largest, cb[6] whether a box plane is NaN) and the
// tiers' counters (tier_words per treelet pass, then a list of node 0 alone
// and its length). The geometry descriptors of a few geometries come with
// the launch.
constexpr int kTierWords = 4;  // bottom roots, middle roots, list space of the middle and of the top tier
constexpr int kTierCounters = kTierWords * kTreeletRounds + 2;
constexpr int kTopRoot = kTierWords * kTreeletRounds, kTopCount = kTopRoot + 1;
constexpr uint32_t kGeomArgs = 8;
struct GeomArgs {
    GeomDesc g[kGeomArgs];
};
__global__ __launch_bounds__(64) void k_build_init(uint32_t* cb, uint32_t* tiers, GeomArgs args, uint32_t ngeom,
                                                   GeomDesc* geoms) {
    const uint32_t t = threadIdx.x;
    if (t < 7) cb[t] = t < 3 ? 0xffffffffu : 0u;
    if (t < kTierCounters) tiers[t] = t == kTopCount ? 1u : 0u;
#pragma unroll
    for (uint32_t k = 0; k < kGeomArgs; ++k)
        if (k == t && k < ngeom) geoms[k] = args.g[k];
}

// Record and box of triangle i.
__device__ inline void make_tri(const GeomDesc* geoms, uint32_t ngeom, uint32_t i, TriRec& r, Box& b,
                                uint32_t* status) {
    uint32_t lo = 0, hi = ngeom;  // last geometry with first_tri <= i
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (geoms[mid].first_tri <= i) lo = mid;
        else hi = mid;
    }
    const GeomDesc g = geoms[lo];
    uint32_t t = i - g.first_tri;
    uint32_t i0 = g.indices[3ull * t], i1 = g.indices[3ull * t + 1], i2 = g.indices[3ull * t + 2];
    if (i0 > g.max_vertex || i1 > g.max_vertex || i2 > g.max_vertex) {
        atomicOr(status, (uint32_t)kStatusBadIndex);
        i0 = i1 = i2 = 0;
    }
    const float* a = reinterpret_cast<const float*>(g.vertices + (uint64_t)i0 * g.stride);
    const float* bb = reinterpret_cast<const float*>(g.vertices + (uint64_t)i1 * g.stride);
    const float* cc = reinterpret_cast<const float*>(g.vertices + (uint64_t)i2 * g.stride);
    float A[3] = {a[0], a[1], a[2]}, B[3] = {bb[0], bb[1], bb[2]}, Cv[3] = {cc[0], cc[1], cc[2]};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.v0[k] = A[k];
        r.v1[k] = B[k];
        r.v2[k] = Cv[k];
        b.lo[k] = mins(mins(A[k], B[k]), Cv[k]);
        b.hi[k] = maxs(maxs(A[k], B[k]), Cv[k]);
    }
    r.prim = t;
    r.geom = lo | ((g.flags & RTG_GEOMETRY_OPAQUE) ? 0u : kNonOpaqueBit);
    r.pad = 0;
}

__device__ inline bool box_has_nan(const Box& b) {
    bool nan = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) nan = nan || b.lo[k] != b.lo[k] || b.hi[k] != b.hi[k];
    return nan;
}

// Triangle records, primitive boxes, centre bounds.
__global__ __launch_bounds__(kSetupThreads) void k_tri_setup(const GeomDesc* geoms, uint32_t ngeom, uint32_t ntri,
                                                             TriRec* tris, Box* boxes, uint32_t* cb,
                                                             uint32_t* status) {
    CentreBounds c;
    for (uint32_t i = blockIdx.x * kSetupThreads + threadIdx.x; i < ntri; i += gridDim.x * kSetupThreads) {
        TriRec r;
        Box b;
        make_tri(geoms, ngeom, i, r, b, status);
        tris[i] = r;
        boxes[i] = b;
        if (box_has_nan(b)) atomicOr(&cb[6], 1u);
        c.add(b);
    }
    reduce_centre_bounds<kSetupThreads>(c, cb);
}

__device__ inline bool registry_has(const uint64_t* reg, uint32_t n, uint64_t a) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        if (reg[mid] < a) lo = mid + 1;
        else hi = mid;
    }
    return lo < n && reg[lo] == a;
}

// World box of an instance: the 8 corners of its BLAS root box through the
// object-to-world transform; empty for an empty or unknown BLAS.
__device__ inline Box instance_world_box(const rtg_instance& in, const AsHeader* bh) {
    Box r = box_empty();
    if (bh == nullptr || bh->prim_count == 0) return r;
    float m[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = (&in.transform[0][0])[k];
    for (int c = 0; c < 8; ++c) {
        V3 p = v3((c & 1) ? bh->hi[0] : bh->lo[0], (c & 2) ? bh->hi[1] : bh->lo[1], (c & 4) ? bh->hi[2] : bh->lo[2]);
        V3 w = m34_point(m, p);
        r.lo[0] = mins(r.lo[0], w.x);
        r.hi[0] = maxs(r.hi[0], w.x);
        r.lo[1] = mins(r.lo[1], w.y);
        r.hi[1] = maxs(r.hi[1], w.y);
        r.lo[2] = mins(r.lo[2], w.z);
        r.hi[2] = maxs(r.hi[2], w.z);
    }
    return r;
}

__device__ inline void fill_inst_rec(InstRec& rec, const rtg_instance& in, uint32_t index, uint64_t blas) {
    float m[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = (&in.transform[0][0])[k];
    m34_inverse(m, rec.w2o);
    rec.blas = blas;
    rec.index = index;
    rec.mask_flags = (in.custom_index_and_mask >> 24) | ((in.sbt_offset_and_flags >> 24) << 8);
}

__device__ inline const AsHeader* checked_blas(const rtg_instance& in, const uint64_t* reg, uint32_t nreg,
                                               uint32_t* status) {
    uint64_t a = in.acceleration_structure_reference;
    if (a == 0) return nullptr;
    if (!registry_has(reg, nreg, a)) {
        atomicOr(status, (uint32_t)kStatusBadBlas);
        return nullptr;
    }
    return reinterpret_cast<const AsHeader*>(a);
}

// Leaf record and world box of instance i.
__device__ inline void make_inst(const rtg_instance* inst, uint32_t i, const uint64_t* reg, uint32_t nreg, InstRec& r,
                                 Box& b, uint32_t* status) {
    rtg_instance in = inst[i];
    const AsHeader* bh = checked_blas(in, reg, nreg, status);
    b = instance_world_box(in, bh);
    fill_inst_rec(r, in, i, bh ? in.acceleration_structure_reference : 0);
}

__global__ __launch_bounds__(256) void k_inst_setup(const rtg_instance* inst, uint32_t n, const uint64_t* reg,
                                                    uint32_t nreg, InstRec* recs, Box* boxes, uint32_t* cb,
                                                    uint32_t* status) {
    CentreBounds c;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        InstRec r;
        Box b;
        make_inst(inst, i, reg, nreg, r, b, status);
        recs[i] = r;
        boxes[i] = b;
        c.add(b);
    }
    reduce_centre_bounds<256>(c, cb);
}

__device__ inline uint32_t spread3(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}
__device__ inline uint32_t quantize10(float c, float lo, float hi) {
    float ext = hi - lo;
    float f = ext > 0.0f ? (c - lo) / ext : 0.0f;
    float q = fminf(fmaxf(f * 1024.0f, 0.0f), 1023.0f);
    return (uint32_t)q;
}

__device__ inline void bounds_from_words(const uint32_t* cb, float lo[3], float hi[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = cb[a] == 0xffffffffu ? __builtin_inff() : ord2f(cb[a]);
        hi[a] = cb[3 + a] == 0u ? -__builtin_inff() : ord2f(cb[3 + a]);
    }
}
__device__ inline uint32_t morton(const Box& b, const float lo[3], const float hi[3]) {
    return (spread3(quantize10(centre(b, 0), lo[0], hi[0])) << 2) |
           (spread3(quantize10(centre(b, 1), lo[1], hi[1])) << 1) | spread3(quantize10(centre(b, 2), lo[2], hi[2]));
}

__global__ __launch_bounds__(256) void k_morton(const Box* boxes, uint32_t n, const uint32_t* cb, uint32_t* keys,
                                                uint32_t* vals) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float lo[3], hi[3];
    bounds_from_words(cb, lo, hi);
    keys[i] = morton(boxes[i], lo, hi);
    vals[i] = i;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort, 8-bit digits, tiles of 256 threads x 8 keys.
// ---------------------------------------------------------------------------
constexpr int kRsThreads = 256;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsThreads * kRsItems;
// Up to this many tiles (262,144 keys) a scatter workgroup sums the tiles'
// counts itself; beyond, a kernel between the two scans them. Builds without
// treelets, summing themselves / with the scan: 60,000 triangles 238 / 244 us,
// 100,000 253 / 256, 130,000 267 / 267, 160,000 278 / 271, 200,000 288 / 284,
// 262,144 303 / 293, 300,000 321 / 307, 500,000 395 / 365. The two cross near
// 130,000, so between there and this line the scan would save 1 to 3 %.
constexpr uint32_t kRsSelfTiles = 128;

// SELF: the counts tile by tile, else digit by digit.
template <bool SELF>
__global__ __launch_bounds__(kRsThreads) void k_rs_hist(const uint32_t* keys, uint32_t n, int shift, uint32_t* hist,
                                                         uint32_t ntiles) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kRsTile + threadIdx.x;
    uint32_t key[kRsItems];
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) key[r] = base + r * kRsThreads < n ? keys[base + r * kRsThreads] : 0u;
#pragma unroll
    for (int r = 0; r < kRsItems; ++r)
        if (base + r * kRsThreads < n) atomicAdd(&h[(key[r] >> shift) & 0xffu], 1u);
    __syncthreads();
    hist[SELF ? (size_t)blockIdx.x * 256 + threadIdx.x : (size_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// Exclusive scan of each digit's counts over the tiles (one workgroup per
// digit) and the digits' totals.
__global__ __launch_bounds__(256) void k_rs_scan(uint32_t* hist, uint32_t ntiles, uint32_t* totals) {
    __shared__ uint32_t part[4];
    uint32_t* row = hist + (size_t)blockIdx.x * ntiles;
    uint32_t run = 0;
    for (uint32_t b = 0; b < ntiles; b += 256) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = i < ntiles ? row[i] : 0u;
        uint32_t total;
        const uint32_t incl = block_scan<256>(v, part, total);
        if (i < ntiles) row[i] = run + incl - v;
        run += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

// A tile's keys to their places. Each wave ranks a run of kRsItems * 64
// consecutive keys against its own counts, 64 at a time, with no barrier in
// between and all of its keys loaded ahead; then the waves' counts become
// first places: 8.3 us a pass over 81,920 keys, bound by the chain of the
// eight ranks, where three barriers and a load per 256 keys and tiles of 4,096
// took 16.8 (a build of 82,000 triangles without treelets 538 -> 467 us).
template <bool SELF>
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(const uint32_t* kin, const uint32_t* vin, uint32_t* kout,
                                                            uint32_t* vout, uint32_t n, int shift,
                                                            const uint32_t* hist, uint32_t ntiles,
                                                            const uint32_t* totals) {
    constexpr int kWaves = kRsThreads / 64;
    static_assert(kRsThreads == 256, "a thread per digit");
    __shared__ uint32_t part[kWaves];
    __shared__ uint32_t wave_cnt[kWaves][256];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t first = blockIdx.x * kRsTile + w * (64 * kRsItems) + lane;
    uint32_t key[kRsItems], val[kRsItems], rank[kRsItems];
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const bool valid = first + r * 64 < n;
        key[r] = valid ? kin[first + r * 64] : 0u;
        val[r] = valid ? vin[first + r * 64] : 0u;
    }
    // first position of each digit in the tile: the totals of the digits
    // below it and its counts in the tiles before
    uint32_t place = 0, mine = 0;
    if (SELF) {
#pragma unroll 8
        for (uint32_t t = 0; t < ntiles; ++t) {
            const uint32_t c = hist[(size_t)t * 256 + threadIdx.x];
            mine += c;
            place += t < blockIdx.x ? c : 0u;
        }
    } else {
        mine = totals[threadIdx.x];
        place = hist[(size_t)threadIdx.x * ntiles + blockIdx.x];
    }
    uint32_t all;
    place += block_scan<256>(mine, part, all) - mine;
    for (int k = 0; k < kWaves; ++k) wave_cnt[k][threadIdx.x] = 0;
    __syncthreads();
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const bool valid = first + r * 64 < n;
        const uint32_t digit = (key[r] >> shift) & 0xffu;
        // lanes of this wave holding the same digit
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const uint64_t bal = __ballot((digit >> bit) & 1u);
            peers &= ((digit >> bit) & 1u) ? bal : ~bal;
        }
        const uint32_t before = wave_cnt[w][digit];
        rank[r] = before + (uint32_t)__popcll(peers & lt_mask);
        wave_order();
        if (valid && (peers & lt_mask) == 0) wave_cnt[w][digit] = before + (uint32_t)__popcll(peers);
        wave_order();
    }
    __syncthreads();
    for (int k = 0; k < kWaves; ++k) {
        const uint32_t c = wave_cnt[k][threadIdx.x];
        wave_cnt[k][threadIdx.x] = place;
        place += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        if (first + r * 64 < n) {
            const uint32_t dst = wave_cnt[w][(key[r] >> shift) & 0xffu] + rank[r];
            kout[dst] = key[r];
            vout[dst] = val[r];
        }
    }
}

// ---------------------------------------------------------------------------
// Radix tree (Karras 2012, Figure 4)
// ---------------------------------------------------------------------------
__device__ inline int delta(const uint32_t* keys, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint32_t a = keys[i], b = keys[j];
    if (a == b) return 32 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clz((int)(a ^ b));
}

// Internal node i of the radix tree over sorted codes: its children's
// references, primitive counts, and its own count.
__device__ inline uint32_t radix_node(const uint32_t* keys, int n, int i, uint32_t child[2], uint32_t count[2]) {
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + (d < 0 ? d : 0);
    int lo = min(i, j), hi = max(i, j);
    child[0] = (lo == gamma) ? (kLeafBit | (uint32_t)gamma) : (uint32_t)gamma;
    child[1] = (hi == gamma + 1) ? (kLeafBit | (uint32_t)(gamma + 1)) : (uint32_t)(gamma + 1);
    count[0] = (uint32_t)(gamma - lo + 1);
    count[1] = (uint32_t)(hi - gamma);
    return (uint32_t)(hi - lo + 1);
}

// The radix tree, the leaf boxes in sorted order and the first pass's tiers.
__global__ __launch_bounds__(kRootThreads) void k_karras(const uint32_t* keys, int n, const uint32_t* order,
                                                         const Box* boxes, Box* lbox, BinNode* bin, uint32_t* rcount,
                                                         uint32_t* low, uint32_t* mid, uint32_t* counts) {
    __shared__ RootList R;
    R.clear();
    const int i = blockIdx.x * kRootThreads + threadIdx.x;
    if (i < n) lbox[i] = boxes[order[i]];
    if (i < n - 1) {
        uint32_t child[2], count[2];
        const uint32_t c = radix_node(keys, n, i, child, count);
        bin[i] = BinNode{child[0], child[1], 0.0f, 0.0f};
        rcount[i] = c;
        tier_roots((uint32_t)i, c, child, count, [&](int tier, uint32_t k) { R.add(tier, k); });
    }
    R.write(low, mid, counts);
}

// ---------------------------------------------------------------------------
// Up to kSmallBuild primitives: one workgroup makes the records, sorts the
// codes in LDS and writes the binary tree. A launch of many workgroups per
// step would be 15 launches of 2 to 5 us each, whatever the count.
// ---------------------------------------------------------------------------
constexpr uint32_t kSmallBuild = 8192;
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr int kSmallItems = kSmallBuild / kSmallThreads;

struct SmallSort {
    uint32_t key[kSmallBuild];
    uint16_t val[kSmallBuild];
    uint16_t cnt[kSmallWaves][256];
    uint32_t part[kSmallWaves];
    uint32_t bounds[8];
    uint32_t tiers[2];
};

struct SmallOut {
    Box* boxes;
    Box* lbox;
    uint32_t* order;
    BinNode* bin;
    uint32_t* rcount;
    uint32_t *low, *mid, *counts, *cb;
};

__device__ inline void small_tree(SmallSort& Z, uint32_t n, const CentreBounds& cb, const SmallOut& O) {
    const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        uint32_t l = cb.lo[a], h = cb.hi[a];
        for (int off = 32; off > 0; off >>= 1) {
            l = min(l, (uint32_t)__shfl_xor((int)l, off));
            h = max(h, (uint32_t)__shfl_xor((int)h, off));
        }
        if (lane == 0) {
            atomicMin(&Z.bounds[a], l);
            atomicMax(&Z.bounds[3 + a], h);
        }
    }
    __syncthreads();
    // wave w holds positions [w * 64 J, (w + 1) * 64 J) of every pass
    const uint32_t J = (n + kSmallThreads - 1) / kSmallThreads;
    const uint32_t first = w * 64 * J + lane;
    uint32_t key[kSmallItems], val[kSmallItems], rank[kSmallItems];
    {
        float lo[3], hi[3];
        bounds_from_words(Z.bounds, lo, hi);
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)kSmallItems; ++j) {
            const uint32_t p = first + j * 64;
            key[j] = val[j] = 0;
            if (j < J && p < n) {
                key[j] = morton(O.boxes[p], lo, hi);
                val[j] = p;
            }
        }
    }
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int shift = 0; shift < 32; shift += 8) {
#pragma unroll
        for (int k = 0; k < 4; ++k) Z.cnt[w][lane + 64 * k] = 0;
        wave_order();
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)kSmallItems; ++j) {
            if (j >= J) break;
            const bool valid = first + j * 64 < n;
            const uint32_t digit = (key[j] >> shift) & 0xffu;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                const uint64_t bal = __ballot((digit >> bit) & 1u);
                peers &= ((digit >> bit) & 1u) ? bal : ~bal;
            }
            const uint32_t before = (uint32_t)__popcll(peers & lt);
            uint32_t run = 0;
            if (valid) run = Z.cnt[w][digit];
            rank[j] = run + before;
            wave_order();
            if (valid && before == 0) Z.cnt[w][digit] = (uint16_t)(run + (uint32_t)__popcll(peers));
            wave_order();
        }
        __syncthreads();
        {
            // exclusive scan over (digit, wave): four waves' counts per thread
            const uint32_t d = t >> 2, w0 = (t & 3u) * 4;
            uint32_t c[4], sum = 0, total;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                c[k] = Z.cnt[w0 + k][d];
                sum += c[k];
            }
            uint32_t run = block_scan<kSmallThreads>(sum, Z.part, total) - sum;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                Z.cnt[w0 + k][d] = (uint16_t)run;
                run += c[k];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)kSmallItems; ++j) {
            if (j >= J) break;
            if (first + j * 64 < n) {
                const uint32_t dst = Z.cnt[w][(key[j] >> shift) & 0xffu] + rank[j];
                Z.key[dst] = key[j];
                Z.val[dst] = (uint16_t)val[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)kSmallItems; ++j) {
            if (j >= J) break;
            const uint32_t p = first + j * 64;
            if (p < n) {
                key[j] = Z.key[p];
                val[j] = Z.val[p];
            }
        }
        // the next pass writes Z.key and Z.val only after two barriers
    }
    for (uint32_t j = 0; j < J; ++j) {
        const uint32_t p = first + j * 64;
        if (p < n) {
            const uint32_t v = Z.val[p];
            O.order[p] = v;
            O.lbox[p] = O.boxes[v];
        }
        if (p + 1 < n) {
            uint32_t child[2], count[2];
            const uint32_t c = radix_node(Z.key, (int)n, (int)p, child, count);
            O.bin[p] = BinNode{child[0], child[1], 0.0f, 0.0f};
            O.rcount[p] = c;
            tier_roots(p, c, child, count, [&](int tier, uint32_t k) {
                (tier == 0 ? O.low : O.mid)[atomicAdd(&Z.tiers[tier], 1u)] = k;
            });
        }
    }
    __syncthreads();
    if (t < 2) O.counts[t] = Z.tiers[t];
}

__device__ inline void small_init(SmallSort& Z) {
    if (threadIdx.x < 8) Z.bounds[threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u;
    if (threadIdx.x < 2) Z.tiers[threadIdx.x] = 0;
    __syncthreads();
}

__global__ __launch_bounds__(kSmallThreads) void k_small_tris(const GeomDesc* geoms, uint32_t ngeom, uint32_t n,
                                                              TriRec* tris, SmallOut O, uint32_t* status) {
    __shared__ SmallSort Z;
    small_init(Z);
    CentreBounds cb;
    for (uint32_t i = threadIdx.x; i < n; i += kSmallThreads) {
        TriRec r;
        Box b;
        make_tri(geoms, ngeom, i, r, b, status);
        tris[i] = r;
        O.boxes[i] = b;
        if (box_has_nan(b)) atomicOr(&O.cb[6], 1u);
        cb.add(b);
    }
    small_tree(Z, n, cb, O);
}

__global__ __launch_bounds__(kSmallThreads) void k_small_insts(const rtg_instance* inst, uint32_t n,
                                                               const uint64_t* reg, uint32_t nreg, InstRec* recs,
                                                               SmallOut O, uint32_t* status) {
    __shared__ SmallSort Z;
    small_init(Z);
    CentreBounds cb;
    for (uint32_t i = threadIdx.x; i < n; i += kSmallThreads) {
        InstRec r;
        Box b;
        make_inst(inst, i, reg, nreg, r, b, status);
        recs[i] = r;
        O.boxes[i] = b;
        cb.add(b);
    }
    small_tree(Z, n, cb, O);
}

// The single node of a structure with at most leaf_max primitives: one leaf
// of all of them in input order (or none).
__global__ void k_wide_single(const Box* boxes, uint32_t n, Node* nodes, uint32_t* order, uint32_t* off,
                              CollapseState* state) {
    if (threadIdx.x == 0) {
        off[0] = 0;
        off[1] = 1;
        *state = CollapseState{1u, 1u, 1u, 0u};
        Node nd;
        const uint32_t ref = n ? (kLeafBit | ((n - 1) << 27)) : kEmpty;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            nd.child[s] = s == 0 ? ref : kEmpty;
            nd.pad[s] = 0;
            set_slot(nd, s, s == 0 ? ref_box(nullptr, ref, boxes, nullptr) : box_empty());
        }
        nodes[0] = nd;
    }
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) order[k] = k;
}

// Slot boxes of the wide nodes of a level (the levels below are done): the
// fold by its definition, for structures with a NaN box plane.
__global__ __launch_bounds__(256) void k_wide_boxes(uint32_t lb, uint32_t m, Node* nodes, const Box* boxes,
                                                    const uint32_t* order) {
    uint32_t w = blockIdx.x * 256 + threadIdx.x;
    if (w >= m) return;
    Node& nd = nodes[lb + w];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        set_slot(nd, k, ref_box(nodes, nd.child[k], boxes, order));
        nd.pad[k] = 0;
    }
}

// Where the parts of a blob lie (bytes from its start).
struct Layout {
    uint64_t nodes_off, prims_off, extra_off, level_off, leafbox_off, total;
    uint32_t node_count;
};

__device__ inline void write_header(uint8_t* blob, const Layout& L, const Node* nodes, uint32_t kind,
                                    uint32_t prim_count, uint32_t geom_count, uint32_t levels) {
    AsHeader hd;
    memset(&hd, 0, sizeof(hd));
    hd.magic = kMagic;
    hd.kind = kind;
    hd.node_count = L.node_count;
    hd.prim_count = prim_count;
    hd.geom_count = geom_count;
    hd.max_depth = levels;
    hd.node_width = 4;
    hd.flags = 0;
    Box r = node_box(nodes[0]);
    for (int a = 0; a < 3; ++a) {
        hd.lo[a] = r.lo[a];
        hd.hi[a] = r.hi[a];
    }
    hd.nodes_off = L.nodes_off;
    hd.prims_off = L.prims_off;
    hd.extra_off = L.extra_off;
    hd.level_off = L.level_off;
    hd.total_size = L.total;
    hd.leafbox_off = L.leafbox_off;
    *reinterpret_cast<AsHeader*>(blob) = hd;
}

// Copies `bytes` (a multiple of sizeof(T)) over the whole grid, T by T.
template <class T>
__device__ inline void grid_copy(void* dst, const void* src, uint64_t bytes) {
    const uint64_t count = bytes / sizeof(T), step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < count; i += step)
        static_cast<T*>(dst)[i] = static_cast<const T*>(src)[i];
}
// Records of `words` T each, out[k] = in[order[k]].
template <class T, uint32_t Words>
__device__ inline void grid_gather(void* dst, const void* src, const uint32_t* order, uint32_t n) {
    const uint64_t count = (uint64_t)n * Words, step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < count; i += step) {
        const uint32_t k = (uint32_t)(i / Words), w = (uint32_t)(i % Words);
        static_cast<T*>(dst)[i] = static_cast<const T*>(src)[(uint64_t)order[k] * Words + w];
    }
}
// Zeroes the 4-byte words of [from, to) (at most 64 bytes of padding).
__device__ inline void zero_pad(uint8_t* blob, uint64_t from, uint64_t to) {
    if (blockIdx.x != 0) return;
    for (uint64_t o = from + 4ull * threadIdx.x; o < to; o += 4ull * blockDim.x)
        *reinterpret_cast<uint32_t*>(blob + o) = 0u;
}

// The blob of a BLAS, and a new version of the registry with its address.
__global__ __launch_bounds__(256) void k_finish_blas(uint8_t* blob, Layout L, const Node* nodes, const TriRec* tris,
                                                     const uint32_t* order, const GeomDesc* geoms, uint32_t ngeom,
                                                     uint32_t n, uint32_t levels, const uint64_t* reg, uint32_t nreg,
                                                     uint64_t* new_reg) {
    grid_copy<uint4>(blob + L.nodes_off, nodes, (uint64_t)L.node_count * sizeof(Node));
    grid_gather<uint4, sizeof(TriRec) / 16>(blob + L.prims_off, tris, order, n);
    if (blockIdx.x != 0) return;
    zero_pad(blob, L.prims_off + (uint64_t)n * sizeof(TriRec), L.extra_off);
    zero_pad(blob, L.extra_off + 4ull * ngeom, L.total);
    uint32_t* gflags = reinterpret_cast<uint32_t*>(blob + L.extra_off);
    for (uint32_t g = threadIdx.x; g < ngeom; g += blockDim.x) gflags[g] = geoms[g].flags;
    if (threadIdx.x == 0) write_header(blob, L, nodes, kKindBlas, n, ngeom, levels);
    const uint64_t addr = reinterpret_cast<uint64_t>(blob);
    for (uint32_t k = threadIdx.x; k < nreg; k += blockDim.x) {
        const uint64_t a = reg[k];
        new_reg[a < addr ? k : k + 1] = a;
        if (a < addr && (k + 1 == nreg || reg[k + 1] > addr)) new_reg[k + 1] = addr;
    }
    if (threadIdx.x == 0 && (nreg == 0 || reg[0] > addr)) new_reg[0] = addr;
}

__global__ __launch_bounds__(256) void k_finish_tlas(uint8_t* blob, Layout L, const Node* nodes, const InstRec* recs,
                                                     const uint32_t* order, const rtg_instance* inst, const Box* lbox,
                                                     const uint32_t* off, uint32_t n, uint32_t levels) {
    grid_copy<uint4>(blob + L.nodes_off, nodes, (uint64_t)L.node_count * sizeof(Node));
    grid_gather<uint4, sizeof(InstRec) / 16>(blob + L.prims_off, recs, order, n);
    // the caller's records: 8-byte words, their alignment
    grid_copy<uint64_t>(blob + L.extra_off, inst, (uint64_t)n * sizeof(rtg_instance));
    grid_copy<uint64_t>(blob + L.leafbox_off, lbox, (uint64_t)n * sizeof(Box));
    if (blockIdx.x != 0) return;
    uint32_t* lv = reinterpret_cast<uint32_t*>(blob + L.level_off);
    for (uint32_t k = threadIdx.x; k < levels + 2; k += blockDim.x) lv[k] = k == 0 ? levels : off[k - 1];
    zero_pad(blob, L.level_off + 4ull * (levels + 2), L.leafbox_off);
    zero_pad(blob, L.leafbox_off + (uint64_t)n * sizeof(Box), L.total);
    if (threadIdx.x == 0) write_header(blob, L, nodes, kKindTlas, n, 0u, levels);
}

// In-place TLAS UPDATE (src/util_structs.rs:285-357): new instance records,
// same topology, slot boxes again from the deepest level up. Instance k's
// record waits on a chain of dependent loads (its index, the caller's
// record, the registry, the BLAS header), so it pays to have all chains in
// flight: one workgroup going through 20,000 instances took 350 us, a lane
// each in as many workgroups as they need 6 us. The registry goes to LDS
// first (a binary search per instance).
constexpr uint32_t kRegistryLds = 1024;

struct TlasParts {
    AsHeader* h;
    Node* nodes;
    InstRec* recs;
    rtg_instance* src;
    Box* leafbox;
};
__device__ inline TlasParts tlas_parts(uint8_t* base) {
    AsHeader* h = reinterpret_cast<AsHeader*>(base);
    return TlasParts{h, reinterpret_cast<Node*>(base + h->nodes_off), reinterpret_cast<InstRec*>(base + h->prims_off),
                     reinterpret_cast<rtg_instance*>(base + h->extra_off),
                     reinterpret_cast<Box*>(base + h->leafbox_off)};
}
__device__ inline const uint64_t* registry_to_lds(const uint64_t* reg, uint32_t nreg, uint64_t* lds) {
    if (nreg > kRegistryLds) return reg;
    for (uint32_t k = threadIdx.x; k < nreg; k += blockDim.x) lds[k] = reg[k];
    return lds;
}
__device__ inline void refit_inst(const TlasParts& P, uint32_t k, const rtg_instance* inst, const uint64_t* reg,
                                  uint32_t nreg, uint32_t* status) {
    uint32_t s = P.recs[k].index;
    rtg_instance in = inst[s];
    const AsHeader* bh = checked_blas(in, reg, nreg, status);
    InstRec r;
    fill_inst_rec(r, in, s, bh ? in.acceleration_structure_reference : 0);
    P.recs[k] = r;
    P.leafbox[k] = instance_world_box(in, bh);
    P.src[s] = in;
}
// Slot i & 3 of node i >> 2 (the levels below are done).
__device__ inline void refit_slot(const TlasParts& P, uint32_t i) {
    Node& nd = P.nodes[i >> 2];
    const uint32_t s = i & 3u;
    set_slot(nd, s, ref_box(P.nodes, nd.child[s], P.leafbox, nullptr));
}
__device__ inline void refit_bounds(const TlasParts& P) {
    if (threadIdx.x != 0) return;
    Box r = node_box(P.nodes[0]);
    for (int a = 0; a < 3; ++a) {
        P.h->lo[a] = r.lo[a];
        P.h->hi[a] = r.hi[a];
    }
}

// The whole update in one workgroup of 256 lanes, one wave per SIMD: while
// another frame's traversal waves fill the GPU, such a workgroup finds room
// on a CU long before a 1024-lane one (four waves per SIMD) would.
__global__ __launch_bounds__(256) void k_tlas_refit(uint8_t* base, const rtg_instance* inst, uint32_t n,
                                                    const uint64_t* reg, uint32_t nreg, uint32_t* status) {
    __shared__ uint64_t s_reg[kRegistryLds];
    const TlasParts P = tlas_parts(base);
    reg = registry_to_lds(reg, nreg, s_reg);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) refit_inst(P, k, inst, reg, nreg, status);
    __syncthreads();
    const uint32_t* lv = reinterpret_cast<const uint32_t*>(base + P.h->level_off);
    const uint32_t levels = lv[0];
    const uint32_t* offs = lv + 1;
    for (uint32_t L = levels; L-- > 0;) {
        for (uint32_t i = 4 * offs[L] + threadIdx.x; i < 4 * offs[L + 1]; i += blockDim.x) refit_slot(P, i);
        __syncthreads();
    }
    refit_bounds(P);
}

__global__ __launch_bounds__(256) void k_refit_insts(uint8_t* base, const rtg_instance* inst, uint32_t n,
                                                     const uint64_t* reg, uint32_t nreg, uint32_t* status) {
    __shared__ uint64_t s_reg[kRegistryLds];
    const TlasParts P = tlas_parts(base);
    reg = registry_to_lds(reg, nreg, s_reg);
    __syncthreads();
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k < n) refit_inst(P, k, inst, reg, nreg, status);
}

// Consecutive levels [from, to) in one workgroup, deepest first.
struct LevelArgs {
    uint32_t off[kReportLevels + 1];
};
__global__ __launch_bounds__(1024) void k_refit_levels(uint8_t* base, LevelArgs A, uint32_t from, uint32_t to) {
    const TlasParts P = tlas_parts(base);
    for (uint32_t L = to; L-- > from;) {
        for (uint32_t i = 4 * A.off[L] + threadIdx.x; i < 4 * A.off[L + 1]; i += blockDim.x) refit_slot(P, i);
        __syncthreads();
    }
    if (from == 0) refit_bounds(P);
}

// One level of nodes [first, end).
__global__ __launch_bounds__(256) void k_refit_level(uint8_t* base, uint32_t first, uint32_t end) {
    const TlasParts P = tlas_parts(base);
    const uint32_t i = 4 * first + blockIdx.x * 256 + threadIdx.x;
    if (i < 4 * end) refit_slot(P, i);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static inline uint64_t align64(uint64_t x) { return (x + 63) & ~uint64_t(63); }
static inline unsigned blocks_for(uint64_t n, unsigned bs) { return (unsigned)((n + bs - 1) / bs); }

// Blob layouts for a tree of node_count nodes in `levels` levels.
static Layout blas_layout(uint32_t n, uint32_t ngeom, uint32_t node_count) {
    Layout L;
    L.node_count = node_count;
    L.nodes_off = 128;
    L.prims_off = align64(L.nodes_off + (uint64_t)node_count * sizeof(Node));
    L.extra_off = align64(L.prims_off + (uint64_t)n * 48);
    L.level_off = 0;
    L.leafbox_off = 0;
    L.total = align64(L.extra_off + (uint64_t)ngeom * 4);
    return L;
}

static Layout tlas_layout(uint32_t n, uint32_t node_count, uint32_t levels) {
    Layout L;
    L.node_count = node_count;
    L.nodes_off = 128;
    L.prims_off = align64(L.nodes_off + (uint64_t)node_count * sizeof(Node));
    L.extra_off = align64(L.prims_off + (uint64_t)n * 64);
    L.level_off = align64(L.extra_off + (uint64_t)n * 64);
    L.leafbox_off = align64(L.level_off + 4ull * (2 + levels));
    L.total = align64(L.leafbox_off + (uint64_t)n * 24);
    return L;
}

// Node capacity of a wide tree over n primitives (its node count is at most
// n - 1: every node has two or more slots).
static inline uint32_t node_cap(uint32_t n) { return n >= 2 ? n - 1 : 1; }

// Scratch of a build over n primitives (records of rec_bytes each).
struct BuildBufs {
    GeomDesc* geoms;
    uint8_t* recs;   // unsorted records
    Box *boxes, *lbox, *ibox;  // of primitives, of sorted leaves, of binary nodes
    uint32_t* cb;    // centre bounds and the NaN flag
    uint32_t *ka, *kb, *va, *vb, *hist, *totals;
    BinNode* bin;
    uint32_t *rcount, *low, *mid, *list, *levels, *tiers;
    Node* nodes;
    uint32_t *wroot, *off, *sums;
    uint4* slots;
    CollapseState* state;
    size_t bytes;
};

// Words of a row of a collapse's turn counts (k_wide_level).
static uint32_t sums_stride(uint32_t cap) { return cap / kWideTurn + 8; }
constexpr uint32_t kCollapseSteps = 12;  // levels launched between two looks at the collapse's progress

static BuildBufs carve_build(void* base, uint32_t n, size_t rec_bytes, uint32_t ngeom) {
    Carve c(base);
    BuildBufs b;
    const uint32_t ntiles = std::max(1u, (n + kRsTile - 1) / kRsTile), cap = node_cap(n);
    b.geoms = c.take<GeomDesc>(std::max(1u, ngeom));
    b.recs = c.take<uint8_t>((size_t)n * rec_bytes);
    b.boxes = c.take<Box>(n);
    b.lbox = c.take<Box>(n);
    b.ibox = c.take<Box>(n);
    b.cb = c.take<uint32_t>(8);
    b.ka = c.take<uint32_t>(n);
    b.kb = c.take<uint32_t>(n);
    b.va = c.take<uint32_t>(std::max(1u, n));
    b.vb = c.take<uint32_t>(n);
    b.hist = c.take<uint32_t>((size_t)256 * ntiles);
    b.totals = c.take<uint32_t>(256);
    b.bin = c.take<BinNode>(n);
    b.rcount = c.take<uint32_t>(n);
    b.low = c.take<uint32_t>(n);
    b.mid = c.take<uint32_t>(n / kTierLow + 2);
    b.list = c.take<uint32_t>(n);
    b.levels = c.take<uint32_t>(n);
    b.tiers = c.take<uint32_t>(kTierCounters);
    b.nodes = c.take<Node>(cap);
    b.wroot = c.take<uint32_t>(cap);
    b.slots = c.take<uint4>(cap);
    b.off = c.take<uint32_t>((size_t)cap + kCollapseSteps + 8);
    b.sums = c.take<uint32_t>((size_t)3 * sums_stride(cap));
    b.state = c.take<CollapseState>(1);
    b.bytes = c.off + 4096;
    return b;
}

static size_t build_scratch_bytes(uint32_t n, size_t rec_bytes, uint32_t ngeom) {
    return carve_build(nullptr, n, rec_bytes, ngeom).bytes;
}

// One bottom-up pass (boxes, with treelets when OPT) over the tiers whose
// roots `tiers` counts.
template <bool OPT>
static void launch_pass(const BuildBufs& b, uint32_t n, uint32_t* tiers, int rounds, hipStream_t s) {
    // a bottom subtree holds 170 of at most 256 primitives on average; the
    // grid loops, so that the count can stay on the device
    const unsigned low_grid = std::min(std::max(1u, n / 96), 8192u);
    // Where the CUs hold every subtree at two workgroups each, a subtree's
    // levels are the launch's time, and 512 lanes take them in fewer turns
    // than 256: builds with treelets of 1,000 triangles 1,205 -> 1,044 us,
    // 20,000 1,043 -> 964 (256 / 512 lanes; all from here on with kept
    // blocks), 80,000 1,382 / 1,325, 100,000 1,470 / 1,390, 110,000 1,499 /
    // 1,412. Beyond, the CUs hold more of the smaller workgroups: 120,000
    // take 1,613 us with 256 lanes and 1,773 with 512, 1 M (before kept
    // blocks) 6,150 and 7,730. The subtrees of a count vary with the mesh, so
    // the line lies a quarter below where uniform meshes cross (256 CUs).
    const bool wide = OPT && n <= 80000;
    auto bottom = wide ? k_tree_bottom<OPT, OPT ? 512 : 256> : k_tree_bottom<OPT, 256>;
    hipLaunchKernelGGL(bottom, dim3(low_grid), dim3(wide ? 512 : 256), 0, s, b.bin, b.ibox, b.rcount, b.lbox, b.low,
                       tiers, rounds);
    const GlobalTree T{b.bin, b.ibox, b.rcount, b.lbox};
    if (n > kTierLow) {
        const unsigned mid_grid = n > kTierHigh ? std::min(n / kTierLow, 1024u) : 1u;
        hipLaunchKernelGGL((k_tree_upper<OPT>), dim3(mid_grid), dim3(kUpperThreads), 0, s, T, b.mid, tiers + 1,
                           kTierLow, n, b.list, b.levels, tiers + 2);
    }
    if (n > kTierHigh)
        hipLaunchKernelGGL((k_tree_upper<OPT>), dim3(1), dim3(kUpperThreads), 0, s, T, b.tiers + kTopRoot,
                           b.tiers + kTopCount, kTierHigh, n, b.list, b.levels, tiers + 3);
}

// From the binary radix tree (n > 1) to the wide nodes in b.nodes; the level
// offsets are in b.off.
static int wide_hierarchy(rtg_ctx* ctx, const BuildBufs& b, uint32_t n, int treelet_rounds, hipStream_t s,
                          BuildReport& rep) {
    if (treelet_rounds == 0) {
        launch_pass<false>(b, n, b.tiers, 1, s);
    } else if (n <= kTierLow) {
        launch_pass<true>(b, n, b.tiers, treelet_rounds, s);
    } else {
        for (int round = 0; round < treelet_rounds; ++round) {
            uint32_t* tiers = b.tiers + kTierWords * round;
            if (round > 0)
                hipLaunchKernelGGL(k_tier_roots, dim3(blocks_for(n - 1, kRootThreads)), dim3(kRootThreads), 0, s, n,
                                   b.bin, b.rcount, b.low, b.mid, tiers);
            launch_pass<true>(b, n, tiers, 1, s);
        }
    }
    const WideTree W{b.bin, b.ibox, b.lbox, b.nodes, b.wroot, node_cap(n)};
    // one workgroup emits 1,024 nodes of a level in about 4 us; beyond a few
    // thousand a launch over many workgroups is the faster way
    const bool one = n <= kSmallBuild;
    const unsigned wide_grid = std::min(n / 1024 + 1, kWideBlocks);
    hipLaunchKernelGGL(k_collapse_top, dim3(1), dim3(kCollapseThreads), 0, s, W, one ? n : 2048u, b.off, b.state);
    do {
        if (!one) {
            hipLaunchKernelGGL(k_wide_expand, dim3(wide_grid), dim3(kWideTurn), 0, s, W, b.off, b.state, b.slots,
                               b.sums, sums_stride(W.cap));
            for (uint32_t k = 0; k < kCollapseSteps; ++k)
                hipLaunchKernelGGL(k_wide_level, dim3(wide_grid), dim3(kWideTurn), 0, s, W, b.off, b.state, k, b.slots,
                                   b.sums, sums_stride(W.cap));
            hipLaunchKernelGGL(k_collapse_advance, dim3(1), dim3(64), 0, s, b.off, b.state, kCollapseSteps);
        }
        hipLaunchKernelGGL(k_build_report, dim3(1), dim3(64), 0, s, b.state, b.off, ctx->d_status, b.cb + 6,
                           ctx->build_report);
        RTG_HIP(hipGetLastError());
        RTG_HIP(hipStreamSynchronize(s));
        rep = *ctx->build_report;
    } while (!one && !rep.done);
    RTG_REQUIRE(rep.done && rep.nodes <= node_cap(n), RTG_ERROR_DEVICE, "BVH collapse: %u nodes, capacity %u",
                rep.nodes, node_cap(n));
    if (rep.nan_boxes) {
        std::vector<uint32_t> off(rep.levels + 1);
        RTG_HIP(hipMemcpyAsync(off.data(), b.off, off.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        RTG_HIP(hipStreamSynchronize(s));
        for (uint32_t L = rep.levels; L-- > 0;) {
            const uint32_t m = off[L + 1] - off[L];
            hipLaunchKernelGGL(k_wide_boxes, dim3(blocks_for(m, 256)), dim3(256), 0, s, off[L], m, b.nodes, b.boxes,
                               b.va);
        }
        RTG_HIP(hipGetLastError());
    }
    return RTG_OK;
}

// The radix tree over more than kSmallBuild primitives whose boxes and
// centre bounds are made; the leaf order ends in b.va.
static void radix_tree(const BuildBufs& b, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, 256)), dim3(256), 0, s, b.boxes, n, b.cb, b.ka, b.va);
    const uint32_t ntiles = (n + kRsTile - 1) / kRsTile;
    uint32_t *kin = b.ka, *kout = b.kb, *vin = b.va, *vout = b.vb;
    for (int pass = 0; pass < 4; ++pass) {
        int shift = pass * 8;
        const bool self = ntiles <= kRsSelfTiles;
        hipLaunchKernelGGL((self ? k_rs_hist<true> : k_rs_hist<false>), dim3(ntiles), dim3(kRsThreads), 0, s, kin, n,
                           shift, b.hist, ntiles);
        if (!self) hipLaunchKernelGGL(k_rs_scan, dim3(256), dim3(256), 0, s, b.hist, ntiles, b.totals);
        hipLaunchKernelGGL((self ? k_rs_scatter<true> : k_rs_scatter<false>), dim3(ntiles), dim3(kRsThreads), 0, s, kin,
                           vin, kout, vout, n, shift, b.hist, ntiles, b.totals);
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    // after 4 passes the sorted data is back in (ka, va)
    hipLaunchKernelGGL(k_karras, dim3(blocks_for(n, kRootThreads)), dim3(kRootThreads), 0, s, b.ka, (int)n, b.va,
                       b.boxes, b.lbox, b.bin, b.rcount, b.low, b.mid, b.tiers);
}

// At most one primitive: the single node.
static int single_node(rtg_ctx* ctx, const BuildBufs& b, uint32_t n, hipStream_t s, BuildReport& rep) {
    hipLaunchKernelGGL(k_wide_single, dim3(1), dim3(256), 0, s, b.boxes, n, b.nodes, b.va, b.off, b.state);
    hipLaunchKernelGGL(k_build_report, dim3(1), dim3(64), 0, s, b.state, b.off, ctx->d_status, b.cb + 6,
                       ctx->build_report);
    RTG_HIP(hipGetLastError());
    RTG_HIP(hipStreamSynchronize(s));
    rep = *ctx->build_report;
    return RTG_OK;
}

static SmallOut small_out(const BuildBufs& b) {
    return SmallOut{b.boxes, b.lbox, b.va, b.bin, b.rcount, b.low, b.mid, b.tiers, b.cb};
}

// Largest level that a refit walks in one workgroup with its neighbours
// (1,024 lanes, a lane per slot: about 1.2 us per 256 nodes, a launch 3 us).
constexpr uint32_t kRefitGroupNodes = 768;

// Workgroups of a blob's last kernel: 16 bytes a lane and a few rounds.
static unsigned finish_grid(uint64_t bytes) { return (unsigned)std::min<uint64_t>(bytes / 4096 / 4 + 1, 4096); }

// Room for `count` addresses in the registry arena. Versions are never
// overwritten: work in flight, and a caller's captured refits, read the one
// of their launch until the context goes.
static int registry_room(rtg_ctx* ctx, uint32_t count, uint64_t** out) {
    if (ctx->registry_used + count > ctx->registry_cap || !ctx->registry_arena) {
        const size_t cap = std::max<size_t>(8192, 16 * (size_t)count);
        uint64_t* p = nullptr;
        RTG_HIP(ctx->blobs.allocate(reinterpret_cast<void**>(&p), cap * sizeof(uint64_t)));
        if (ctx->registry_arena) ctx->retired.push_back(ctx->registry_arena);
        ctx->registry_arena = p;
        ctx->registry_cap = cap;
        ctx->registry_used = 0;
    }
    *out = ctx->registry_arena + ctx->registry_used;
    return RTG_OK;
}
static void registry_commit(rtg_ctx* ctx, uint64_t* version, uint32_t count) {
    ctx->d_registry = version;
    ctx->registry_count = count;
    ctx->registry_used += count;
}

int build_report_init(rtg_ctx* ctx) {
    RTG_HIP(hipHostMalloc(reinterpret_cast<void**>(&ctx->build_report), sizeof(BuildReport)));
    return RTG_OK;
}

int refresh_registry(rtg_ctx* ctx) {
    std::vector<uint64_t> addrs;  // ascending, as the map holds them
    for (auto& kv : ctx->structures)
        if (kv.second.kind == kKindBlas) addrs.push_back(kv.first);
    uint64_t* d = nullptr;
    int st = registry_room(ctx, (uint32_t)addrs.size(), &d);
    if (st != RTG_OK) return st;
    if (!addrs.empty()) RTG_HIP(hipMemcpy(d, addrs.data(), addrs.size() * sizeof(uint64_t), hipMemcpyHostToDevice));
    registry_commit(ctx, d, (uint32_t)addrs.size());
    return RTG_OK;
}

int launch_refit(rtg_ctx* ctx, uint8_t* tlas, const std::vector<uint32_t>& level_off, const rtg_instance* instances,
                 uint32_t count, hipStream_t s) {
    LaunchTimer timer(ctx, RTG_KERNEL_REFIT, s);
    const uint32_t levels = level_off.empty() ? 0 : (uint32_t)level_off.size() - 1;
    // one workgroup takes about 4 us per 256 instances, a second launch 3 us
    if (count <= 256 || levels == 0) {
        hipLaunchKernelGGL(k_tlas_refit, dim3(1), dim3(256), 0, s, tlas, instances, count, ctx->d_registry,
                           ctx->registry_count, ctx->d_status);
        RTG_HIP(hipGetLastError());
        return RTG_OK;
    }
    hipLaunchKernelGGL(k_refit_insts, dim3(blocks_for(count, 256)), dim3(256), 0, s, tlas, instances, count,
                       ctx->d_registry, ctx->registry_count, ctx->d_status);
    LevelArgs A = {};
    std::copy(level_off.begin(), level_off.end(), A.off);
    auto nodes = [&](uint32_t L) { return level_off[L + 1] - level_off[L]; };
    for (uint32_t to = levels; to > 0;) {
        // runs of levels that one workgroup walks faster than a launch each
        uint32_t from = to, most = 0;
        while (from > 0 && nodes(from - 1) <= kRefitGroupNodes) most = std::max(most, nodes(--from));
        if (from < to) {
            hipLaunchKernelGGL(k_refit_levels, dim3(1), dim3(most <= 256 ? 256 : 1024), 0, s, tlas, A, from, to);
        } else {
            --from;
            hipLaunchKernelGGL(k_refit_level, dim3(blocks_for(4ull * nodes(from), 256)), dim3(256), 0, s, tlas,
                               level_off[from], level_off[from + 1]);
        }
        to = from;
    }
    RTG_HIP(hipGetLastError());
    return RTG_OK;
}

int check_status(rtg_ctx* ctx, hipStream_t stream, uint32_t mask, const char* what) {
    uint32_t st = 0;
    RTG_HIP(hipStreamSynchronize(stream));
    RTG_HIP(hipMemcpy(&st, ctx->d_status, 4, hipMemcpyDeviceToHost));
    if (st & mask) {
        uint32_t cleared = st & ~mask;
        RTG_HIP(hipMemcpy(ctx->d_status, &cleared, 4, hipMemcpyHostToDevice));
        set_error("%s: device reported status 0x%x (1: index > max_vertex, 2: reference to an unknown BLAS, "
                  "4: traversal stack overflow)",
                  what, st & mask);
        return RTG_ERROR_INVALID_ARGUMENT;
    }
    return RTG_OK;
}

}  // namespace rtg

using namespace rtg;

extern "C" int rtg_blas_query_sizes(rtg_ctx* ctx, const rtg_geometry* geoms, uint32_t n_geom, rtg_build_sizes* out) {
    clear_error();
    RTG_REQUIRE(ctx && out && (geoms || n_geom == 0), RTG_ERROR_INVALID_ARGUMENT, "rtg_blas_query_sizes: null argument");
    uint64_t total = 0;
    for (uint32_t g = 0; g < n_geom; ++g) total += geoms[g].index_count / 3;
    RTG_REQUIRE(total < (1ull << 27), RTG_ERROR_LIMIT, "BLAS has %llu triangles (limit 2^27)",
                (unsigned long long)total);
    // an upper bound: the blob of a build holds its actual node count
    Layout L = blas_layout((uint32_t)total, n_geom, node_cap((uint32_t)total));
    out->acceleration_structure_size = L.total;
    out->build_scratch_size = build_scratch_bytes((uint32_t)total, sizeof(TriRec), n_geom);
    out->update_scratch_size = 0;
    return RTG_OK;
}

extern "C" int rtg_tlas_query_sizes(rtg_ctx* ctx, uint32_t count, rtg_build_sizes* out) {
    clear_error();
    RTG_REQUIRE(ctx && out, RTG_ERROR_INVALID_ARGUMENT, "rtg_tlas_query_sizes: null argument");
    RTG_REQUIRE(count < (1u << 27), RTG_ERROR_LIMIT, "TLAS has %u instances (limit 2^27)", count);
    Layout L = tlas_layout(count, node_cap(count), node_cap(count));
    out->acceleration_structure_size = L.total;
    out->build_scratch_size = build_scratch_bytes(count, sizeof(InstRec), 1);
    out->update_scratch_size = 0;
    return RTG_OK;
}

extern "C" int rtg_blas_build(rtg_ctx* ctx, const rtg_geometry* geoms, uint32_t n_geom, uint32_t flags, rtg_blas* out,
                              void* stream) {
    clear_error();
    RTG_REQUIRE(ctx && out && (geoms || n_geom == 0), RTG_ERROR_INVALID_ARGUMENT, "rtg_blas_build: null argument");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    RTG_HIP(hipSetDevice(ctx->device));
    uint64_t total = 0;
    std::vector<GeomDesc> gd(std::max(1u, n_geom));
    for (uint32_t g = 0; g < n_geom; ++g) {
        const rtg_geometry& G = geoms[g];
        RTG_REQUIRE(G.index_count % 3 == 0, RTG_ERROR_INVALID_ARGUMENT,
                    "geometry %u: index_count %u is not a multiple of 3", g, G.index_count);
        RTG_REQUIRE(G.vertex_stride >= 12 && G.vertex_stride % 4 == 0, RTG_ERROR_INVALID_ARGUMENT,
                    "geometry %u: vertex_stride %u (need >= 12, multiple of 4)", g, G.vertex_stride);
        RTG_REQUIRE(G.index_count == 0 || (G.vertex_data && G.index_data), RTG_ERROR_INVALID_ARGUMENT,
                    "geometry %u: null vertex or index data", g);
        gd[g].vertices = reinterpret_cast<const uint8_t*>(G.vertex_data);
        gd[g].indices = reinterpret_cast<const uint32_t*>(G.index_data);
        gd[g].stride = G.vertex_stride;
        gd[g].max_vertex = G.max_vertex;
        gd[g].first_tri = (uint32_t)total;
        gd[g].flags = G.flags;
        total += G.index_count / 3;
        RTG_REQUIRE(total < (1ull << 27), RTG_ERROR_LIMIT, "BLAS exceeds 2^27 triangles");
    }
    uint32_t n = (uint32_t)total;
    if (ensure_room(ctx, ctx->scratch, build_scratch_bytes(n, sizeof(TriRec), n_geom)) != RTG_OK)
        return RTG_ERROR_OUT_OF_MEMORY;
    const BuildBufs b = carve_build(ctx->scratch.ptr, n, sizeof(TriRec), n_geom);
    GeomArgs args = {};
    const uint32_t by_arg = n_geom <= kGeomArgs ? n_geom : 0;
    std::copy(gd.begin(), gd.begin() + by_arg, args.g);
    hipLaunchKernelGGL(k_build_init, dim3(1), dim3(64), 0, s, b.cb, b.tiers, args, by_arg, b.geoms);
    // the copy source must outlive the asynchronous copy: the build
    // synchronises its stream before returning
    if (n_geom > kGeomArgs)
        RTG_HIP(hipMemcpyAsync(b.geoms, gd.data(), n_geom * sizeof(GeomDesc), hipMemcpyHostToDevice, s));
    TriRec* tris = reinterpret_cast<TriRec*>(b.recs);
    if (n > 1 && n <= kSmallBuild) {
        hipLaunchKernelGGL(k_small_tris, dim3(1), dim3(kSmallThreads), 0, s, b.geoms, n_geom, n, tris, small_out(b),
                           ctx->d_status);
    } else if (n > 0) {
        hipLaunchKernelGGL(k_tri_setup, dim3(std::min(blocks_for(n, kSetupThreads), kSetupBlocks)),
                           dim3(kSetupThreads), 0, s, b.geoms, n_geom, n, tris, b.boxes, b.cb, ctx->d_status);
        if (n > 1) radix_tree(b, n, s);
    }
    BuildReport rep;
    int st = n > 1 ? wide_hierarchy(ctx, b, n, (flags & RTG_BUILD_PREFER_FAST_TRACE) ? kTreeletRounds : 0, s, rep)
                   : single_node(ctx, b, n, s, rep);
    if (st != RTG_OK) {
        hipStreamSynchronize(s);  // pending copies read host memory of this frame
        return st;
    }
    if (rep.status & kStatusBadIndex) return check_status(ctx, s, kStatusBadIndex, "rtg_blas_build");
    const Layout L = blas_layout(n, n_geom, rep.nodes);
    uint64_t* new_reg = nullptr;
    st = registry_room(ctx, ctx->registry_count + 1, &new_reg);
    if (st != RTG_OK) return st;
    void* block = nullptr;
    uint64_t alloc = 0;
    st = ctx->blobs.take(L.total, &block, &alloc);
    if (st != RTG_OK) return st;
    uint8_t* blob = static_cast<uint8_t*>(block);
    hipLaunchKernelGGL(k_finish_blas, dim3(finish_grid(L.total)), dim3(256), 0, s, blob, L, b.nodes, tris, b.va,
                       b.geoms, n_geom, n, rep.levels, ctx->d_registry, ctx->registry_count, new_reg);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        hipFree(blob);
        set_error("rtg_blas_build: %s", hipGetErrorString(e));
        return RTG_ERROR_DEVICE;
    }
    uint64_t addr = reinterpret_cast<uint64_t>(blob);
    ctx->structures[addr] = AsRecord{kKindBlas, n, L.node_count, L.total, alloc, {}};
    registry_commit(ctx, new_reg, ctx->registry_count + 1);
    *out = addr;
    return RTG_OK;
}

extern "C" int rtg_tlas_build(rtg_ctx* ctx, const rtg_instance* instances, uint32_t count, uint32_t flags,
                              rtg_tlas* out, void* stream) {
    clear_error();
    RTG_REQUIRE(ctx && out && (instances || count == 0), RTG_ERROR_INVALID_ARGUMENT, "rtg_tlas_build: null argument");
    RTG_REQUIRE(count < (1u << 27), RTG_ERROR_LIMIT, "TLAS has %u instances (limit 2^27)", count);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    RTG_HIP(hipSetDevice(ctx->device));
    uint32_t n = count;
    if (ensure_room(ctx, ctx->scratch, build_scratch_bytes(n, sizeof(InstRec), 1)) != RTG_OK)
        return RTG_ERROR_OUT_OF_MEMORY;
    const BuildBufs b = carve_build(ctx->scratch.ptr, n, sizeof(InstRec), 1);
    hipLaunchKernelGGL(k_build_init, dim3(1), dim3(64), 0, s, b.cb, b.tiers, GeomArgs{}, 0u, b.geoms);
    InstRec* recs = reinterpret_cast<InstRec*>(b.recs);
    if (n > 1 && n <= kSmallBuild) {
        hipLaunchKernelGGL(k_small_insts, dim3(1), dim3(kSmallThreads), 0, s, instances, n, ctx->d_registry,
                           ctx->registry_count, recs, small_out(b), ctx->d_status);
    } else if (n > 0) {
        hipLaunchKernelGGL(k_inst_setup, dim3(blocks_for(n, 256)), dim3(256), 0, s, instances, n, ctx->d_registry,
                           ctx->registry_count, recs, b.boxes, b.cb, ctx->d_status);
        if (n > 1) radix_tree(b, n, s);
        else hipMemcpyAsync(b.lbox, b.boxes, sizeof(Box), hipMemcpyDeviceToDevice, s);
    }
    BuildReport rep;
    int st = n > 1 ? wide_hierarchy(ctx, b, n, (flags & RTG_BUILD_PREFER_FAST_TRACE) ? kTreeletRounds : 0, s, rep)
                   : single_node(ctx, b, n, s, rep);
    if (st != RTG_OK) {
        hipStreamSynchronize(s);
        return st;
    }
    if (rep.status & kStatusBadBlas) return check_status(ctx, s, kStatusBadBlas, "rtg_tlas_build");
    const Layout L = tlas_layout(n, rep.nodes, rep.levels);
    void* block = nullptr;
    uint64_t alloc = 0;
    st = ctx->blobs.take(L.total, &block, &alloc);
    if (st != RTG_OK) return st;
    uint8_t* blob = static_cast<uint8_t*>(block);
    hipLaunchKernelGGL(k_finish_tlas, dim3(finish_grid(L.total)), dim3(256), 0, s, blob, L, b.nodes, recs, b.va,
                       instances, b.lbox, b.off, n, rep.levels);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        hipFree(blob);
        set_error("rtg_tlas_build: %s", hipGetErrorString(e));
        return RTG_ERROR_DEVICE;
    }
    uint64_t addr = reinterpret_cast<uint64_t>(blob);
    std::vector<uint32_t> level_off;
    if (rep.levels <= kReportLevels) level_off.assign(rep.off, rep.off + rep.levels + 1);
    ctx->structures[addr] = AsRecord{kKindTlas, n, L.node_count, L.total, alloc, level_off};
    *out = addr;
    return RTG_OK;
}

extern "C" int rtg_tlas_refit(rtg_ctx* ctx, rtg_tlas tlas, const rtg_instance* instances, uint32_t count,
                              void* stream) {
    clear_error();
    RTG_REQUIRE(ctx && (instances || count == 0), RTG_ERROR_INVALID_ARGUMENT, "rtg_tlas_refit: null argument");
    auto it = ctx->structures.find(tlas);
    RTG_REQUIRE(it != ctx->structures.end() && it->second.kind == kKindTlas, RTG_ERROR_NOT_FOUND,
                "rtg_tlas_refit: 0x%llx is not a TLAS of this context", (unsigned long long)tlas);
    RTG_REQUIRE(it->second.prim_count == count, RTG_ERROR_INVALID_ARGUMENT,
                "rtg_tlas_refit: %u instances, the TLAS was built with %u", count, it->second.prim_count);
    return launch_refit(ctx, reinterpret_cast<uint8_t*>(tlas), it->second.level_off, instances, count,
                        reinterpret_cast<hipStream_t>(stream));
}

extern "C" int rtg_tlas_clone(rtg_ctx* ctx, rtg_tlas src, rtg_tlas* out, void* stream) {
    clear_error();
    RTG_REQUIRE(ctx && out, RTG_ERROR_INVALID_ARGUMENT, "rtg_tlas_clone: null argument");
    auto it = ctx->structures.find(src);
    RTG_REQUIRE(it != ctx->structures.end() && it->second.kind == kKindTlas, RTG_ERROR_NOT_FOUND,
                "rtg_tlas_clone: 0x%llx is not a TLAS of this context", (unsigned long long)src);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    RTG_HIP(hipSetDevice(ctx->device));
    void* blob = nullptr;
    uint64_t alloc = 0;
    const int st = ctx->blobs.take(it->second.size, &blob, &alloc);
    if (st != RTG_OK) return st;
    RTG_HIP(hipMemcpyAsync(blob, reinterpret_cast<const void*>(src), it->second.size, hipMemcpyDeviceToDevice, s));
    uint64_t addr = reinterpret_cast<uint64_t>(blob);
    AsRecord rec = it->second;
    rec.alloc = alloc;
    ctx->structures[addr] = rec;
    *out = addr;
    return RTG_OK;
}

static int destroy_as(rtg_ctx* ctx, uint64_t addr, uint32_t kind, const char* what) {
    clear_error();
    RTG_REQUIRE(ctx, RTG_ERROR_INVALID_ARGUMENT, "%s: null context", what);
    auto it = ctx->structures.find(addr);
    RTG_REQUIRE(it != ctx->structures.end() && it->second.kind == kind, RTG_ERROR_NOT_FOUND,
                "%s: 0x%llx is not a live structure of this kind", what, (unsigned long long)addr);
    RTG_HIP(hipDeviceSynchronize());
    ctx->blobs.put(reinterpret_cast<void*>(addr), it->second.alloc);
    ctx->structures.erase(it);
    if (kind == kKindBlas) return refresh_registry(ctx);
    return RTG_OK;
}

extern "C" int rtg_blas_destroy(rtg_ctx* ctx, rtg_blas blas) { return destroy_as(ctx, blas, kKindBlas, "rtg_blas_destroy"); }
extern "C" int rtg_tlas_destroy(rtg_ctx* ctx, rtg_tlas tlas) { return destroy_as(ctx, tlas, kKindTlas, "rtg_tlas_destroy"); }

extern "C" int rtg_as_get_info(rtg_ctx* ctx, uint64_t addr, rtg_as_info* out) {
    clear_error();
    RTG_REQUIRE(ctx && out, RTG_ERROR_INVALID_ARGUMENT, "rtg_as_get_info: null argument");
    auto it = ctx->structures.find(addr);
    RTG_REQUIRE(it != ctx->structures.end(), RTG_ERROR_NOT_FOUND, "rtg_as_get_info: unknown structure 0x%llx",
                (unsigned long long)addr);
    AsHeader h;
    RTG_HIP(hipDeviceSynchronize());
    RTG_HIP(hipMemcpy(&h, reinterpret_cast<const void*>(addr), sizeof(h), hipMemcpyDeviceToHost));
    out->kind = h.kind;
    out->node_count = h.node_count;
    out->prim_count = h.prim_count;
    out->geometry_count = h.geom_count;
    out->max_depth = h.max_depth;
    out->node_width = h.node_width;
    for (int a = 0; a < 3; ++a) {
        out->bounds[a] = h.lo[a];
        out->bounds[3 + a] = h.hi[a];
    }
    out->size_bytes = h.total_size;
    return RTG_OK;
}
