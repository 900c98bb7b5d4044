// queue_alloc.hpp -- slots of two device queues for a workgroup of 256 lanes.
// Device code over wave and workgroup operations that includes no HIP header
// itself (include it after one), so that a CPU build can run it under any
// order of the waves.
#pragma once

#include <cstdint>

namespace rtg {

// Allocation from two queues by a whole workgroup (every lane calls it; lanes
// that need nothing pass 0): one atomic per queue and 256 lanes. Atomics to
// one address pass one at a time, about 13 ns each, which bound the shading of
// large images when every wave made its own (7.4 M paths: 115 k of them,
// 1.5 ms). EVEN: every lane wants the same number of entries of the first
// queue or none, so ranks come from a ballot.
//
// A caller allocates once a round. Waves read the totals and bases of a round
// after its last barrier, so a wave may still read them while another is a
// round ahead and writes its total: rounds alternate between two copies. A
// copy's next write comes two rounds later, behind the two barriers of the
// round between, which no wave passes before it has done its reads. (A third
// barrier a round would order one copy as well.)
struct QueueAlloc {
    struct Copy {
        uint32_t total[2][4], base[2];
    } copy[2];
};
__device__ inline uint32_t wave_rank(uint32_t want, bool even, uint32_t& total) {
    const int lane = threadIdx.x & 63;
    if (even) {
        const uint64_t m = __ballot(want != 0u);
        const uint32_t each = m ? (uint32_t)__shfl((int)want, (int)__builtin_ctzll(m)) : 0u;
        total = each * (uint32_t)__popcll(m);
        return each * (uint32_t)__popcll(m & (lane == 0 ? 0ull : (~0ull >> (64 - lane))));
    }
    uint32_t incl = want;
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t v = (uint32_t)__shfl_up((int)incl, off);
        if (lane >= off) incl += v;
    }
    total = (uint32_t)__shfl((int)incl, 63);
    return incl - want;
}
template <bool EVEN>
__device__ inline void block_alloc(QueueAlloc& alloc, uint32_t round, uint32_t want0, uint32_t* counter0, bool want1,
                                   uint32_t* counter1, uint32_t& slot0, uint32_t& slot1) {
    QueueAlloc::Copy& A = alloc.copy[round & 1u];
    const int w = threadIdx.x >> 6;
    uint32_t t0, t1;
    const uint32_t r0 = wave_rank(want0, EVEN, t0), r1 = wave_rank(want1 ? 1u : 0u, true, t1);
    if ((threadIdx.x & 63) == 0) {
        A.total[0][w] = t0;
        A.total[1][w] = t1;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const uint32_t* tt = A.total[threadIdx.x];
        const uint32_t sum = (tt[0] + tt[1]) + (tt[2] + tt[3]);
        A.base[threadIdx.x] = sum ? atomicAdd(threadIdx.x ? counter1 : counter0, sum) : 0u;
    }
    __syncthreads();
    uint32_t b0 = A.base[0], b1 = A.base[1];
    for (int k = 0; k < 3; ++k)
        if (k < w) {
            b0 += A.total[0][k];
            b1 += A.total[1][k];
        }
    slot0 = b0 + r0;
    slot1 = b1 + r1;
}

}  // namespace rtg
