// Runs csrc/queue_alloc.hpp on the CPU, a fiber per lane of one workgroup, with
// the four waves in every order of priority: a wave that can run goes on until
// a barrier stops it, which is as far ahead as the barriers let it get. Slots
// have to be those of some serial order: disjoint, and without gaps.
#include <ucontext.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

namespace sim {
constexpr int kLanes = 256, kWaves = 4;
struct Lane {
    ucontext_t ctx;
    std::vector<char> stack;
    uint64_t ops = 0, barriers = 0;  // wave operations and barriers this lane has reached
    uint64_t need_ops = 0, need_barriers = 0;
    bool done = false;
};
static Lane lanes[kLanes];
static ucontext_t scheduler;
static int current;
static int arrived[kWaves][4096], arrived_barrier[4096];  // lanes that reached the n-th wave operation, barrier
static int64_t posted[2][kLanes];
struct Index {
    uint32_t x;
};

static void yield() { swapcontext(&lanes[current].ctx, &scheduler); }

// All lanes of the wave meet here; `v` is then what each of them posted.
static const int64_t* meet(int64_t mine) {
    Lane& l = lanes[current];
    const int me = current;
    int64_t* row = posted[l.ops & 1];
    row[me] = mine;
    l.need_ops = ++l.ops;
    ++arrived[me >> 6][l.ops];
    yield();
    return row + (me & ~63);
}
static bool runnable(int i) {
    const Lane& l = lanes[i];
    if (l.done) return false;
    return (l.need_ops == 0 || arrived[i >> 6][l.need_ops] == 64) &&
           (l.need_barriers == 0 || arrived_barrier[l.need_barriers] == kLanes);
}
}  // namespace sim

#define __device__
#define threadIdx (sim::Index{(uint32_t)sim::current})
static uint64_t __ballot(bool b) {
    const int64_t* v = sim::meet(b);
    uint64_t m = 0;
    for (int k = 0; k < 64; ++k) m |= (uint64_t)(v[k] != 0) << k;
    return m;
}
static int __shfl(int x, int lane) { return (int)sim::meet(x)[lane]; }
static int __shfl_up(int x, int off) {
    const int lane = sim::current & 63;
    const int64_t* v = sim::meet(x);
    return (int)v[lane >= off ? lane - off : lane];
}
static void __syncthreads() {
    sim::Lane& l = sim::lanes[sim::current];
    l.need_barriers = ++l.barriers;
    ++sim::arrived_barrier[l.barriers];
    sim::yield();
}
static int __popcll(uint64_t x) { return __builtin_popcountll(x); }
static uint32_t atomicAdd(uint32_t* p, uint32_t v) {
    const uint32_t old = *p;
    *p += v;
    return old;
}

#include "queue_alloc.hpp"

static constexpr int kRounds = 5;
static rtg::QueueAlloc g_alloc;
static uint32_t g_counter[2];
static uint32_t g_want[kRounds][sim::kLanes][2], g_slot[kRounds][sim::kLanes][2];
static bool g_even;

static void lane_main() {
    for (uint32_t r = 0; r < kRounds; ++r) {
        const int i = sim::current;
        const uint32_t w0 = g_want[r][i][0];
        const bool w1 = g_want[r][i][1] != 0;
        uint32_t a, b;
        if (g_even) rtg::block_alloc<true>(g_alloc, r, w0, &g_counter[0], w1, &g_counter[1], a, b);
        else rtg::block_alloc<false>(g_alloc, r, w0, &g_counter[0], w1, &g_counter[1], a, b);
        g_slot[r][sim::current][0] = a;
        g_slot[r][sim::current][1] = b;
    }
    sim::lanes[sim::current].done = true;
    sim::yield();
}

static bool run(const int order[4]) {
    g_counter[0] = g_counter[1] = 0;
    for (auto& w : sim::arrived) std::fill(std::begin(w), std::end(w), 0);
    std::fill(std::begin(sim::arrived_barrier), std::end(sim::arrived_barrier), 0);
    for (int i = 0; i < sim::kLanes; ++i) {
        sim::Lane& l = sim::lanes[i];
        l.stack.resize(32768);
        l.ops = l.barriers = l.need_ops = l.need_barriers = 0;
        l.done = false;
        getcontext(&l.ctx);
        l.ctx.uc_stack.ss_sp = l.stack.data();
        l.ctx.uc_stack.ss_size = l.stack.size();
        l.ctx.uc_link = nullptr;
        makecontext(&l.ctx, lane_main, 0);
    }
    while (true) {
        int pick = -1;
        for (int w = 0; w < sim::kWaves && pick < 0; ++w)
            for (int k = 0; k < 64 && pick < 0; ++k)
                if (sim::runnable(64 * order[w] + k)) pick = 64 * order[w] + k;
        if (pick < 0) break;
        sim::current = pick;
        swapcontext(&sim::scheduler, &sim::lanes[pick].ctx);
    }
    for (int i = 0; i < sim::kLanes; ++i)
        if (!sim::lanes[i].done) return std::printf("lane %d never ended\n", i), false;
    for (int q = 0; q < 2; ++q) {
        uint32_t total = 0;
        for (auto& round : g_want)
            for (auto& lane : round) total += lane[q];
        if (total != g_counter[q]) return std::printf("queue %d: %u of %u entries\n", q, g_counter[q], total), false;
        std::vector<char> taken(total, 0);
        for (int r = 0; r < kRounds; ++r)
            for (int i = 0; i < sim::kLanes; ++i)
                for (uint32_t k = 0; k < g_want[r][i][q]; ++k) {
                    const uint32_t s = g_slot[r][i][q] + k;
                    if (s >= total || taken[s])
                        return std::printf("queue %d round %d lane %d: slot %u\n", q, r, i, s), false;
                    taken[s] = 1;
                }
    }
    return true;
}

int main() {
    std::srand(7);
    for (int kind = 0; kind < 4; ++kind) {  // mixed; even; whole waves without; an empty last round
        g_even = kind == 1;
        for (int r = 0; r < kRounds; ++r)
            for (int i = 0; i < sim::kLanes; ++i) {
                uint32_t a = (uint32_t)(std::rand() % 5) * 2, b = (uint32_t)(std::rand() % 3 == 0);
                if (g_even) a = a > 4 ? 4 : 0;
                if (kind == 2 && (i >> 6) % 2 == r % 2) a = b = 0;
                if (kind == 3 && r == kRounds - 1) a = b = 0;
                g_want[r][i][0] = a;
                g_want[r][i][1] = b;
            }
        int order[4] = {0, 1, 2, 3};
        do {
            if (!run(order)) {
                std::printf("kind %d, waves %d %d %d %d\n", kind, order[0], order[1], order[2], order[3]);
                return 1;
            }
        } while (std::next_permutation(order, order + 4));
    }
    std::printf("queue slots: ok\n");
    return 0;
}
