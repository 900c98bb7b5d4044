// flight.hpp -- which of a process's traces are on a GPU. Host code without HIP, so that a
// CPU build can run it.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <mutex>

namespace rtg {

// A frame arena with a trace takes a word: `started` counts the traces the
// host has enqueued on it, and the last kernel of each stores that trace's
// number in `ended` (host memory that the GPU writes). A word has one arena,
// whose traces run one after another, and is given back with it; an arena that
// finds none free is left out, which only changes what others are taken to be.
constexpr int kFlightWords = 256;
struct FlightTable {
    uint32_t* ended = nullptr;

    int take() {
        std::lock_guard<std::mutex> lk(mu);
        for (int k = 0; k < kFlightWords; ++k)
            if (!used[k]) {
                used[k] = true;
                top.store(std::max(top.load(), k + 1));
                return k;
            }
        return -1;
    }
    // of an arena none of whose traces is on the GPU any more
    void give(int word) {
        if (word < 0) return;
        std::lock_guard<std::mutex> lk(mu);
        started[word].store(ended_now(word));
        used[word] = false;
    }
    // enters a trace; its number, which its last kernel stores
    uint32_t start(int word) { return started[word].fetch_add(1) + 1; }
    // words other than `word` with a trace on the GPU (a moment's view)
    int others(int word) const {
        int n = 0;
        for (int k = 0; k < top.load(std::memory_order_relaxed); ++k)
            if (k != word && started[k].load(std::memory_order_relaxed) != ended_now(k)) ++n;
        return n;
    }

private:
    uint32_t ended_now(int k) const { return __atomic_load_n(&ended[k], __ATOMIC_RELAXED); }
    std::mutex mu;
    bool used[kFlightWords] = {};
    std::atomic<int> top{0};  // words that were ever taken come first
    std::atomic<uint32_t> started[kFlightWords] = {};
};

}  // namespace rtg
