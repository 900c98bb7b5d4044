// csrc/flight.hpp on the CPU: each word has one owner at a time, comes back
// with it, and tells of its own traces only.
#include "flight.hpp"

#include <cstdio>
#include <vector>

using rtg::FlightTable;
using rtg::kFlightWords;

#define CHECK(x)                                                \
    do {                                                        \
        if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1; \
    } while (0)

int main() {
    static uint32_t ended[kFlightWords];
    static FlightTable T;
    T.ended = ended;
    std::vector<int> w;
    for (int k = 0; k < kFlightWords; ++k) {
        w.push_back(T.take());
        for (int j = 0; j < k; ++j) CHECK(w[j] != w[k]);
        CHECK(w[k] >= 0 && w[k] < kFlightWords);
    }
    CHECK(T.take() == -1);
    CHECK(T.others(-1) == 0);
    // a trace is seen by all but its own arena, until it ends
    const uint32_t a = T.start(w[3]), b = T.start(w[7]);
    CHECK(T.others(-1) == 2 && T.others(w[3]) == 1 && T.others(w[7]) == 1 && T.others(w[9]) == 2);
    ended[w[7]] = b;
    CHECK(T.others(w[9]) == 1 && T.others(w[3]) == 0 && T.others(w[7]) == 1);
    // two in a row on one arena: in flight until the second has ended
    const uint32_t a2 = T.start(w[3]);
    ended[w[3]] = a;
    CHECK(T.others(w[9]) == 1);
    ended[w[3]] = a2;
    CHECK(T.others(w[9]) == 0);
    // a word given back and taken again starts anew, whatever was left in it
    T.start(w[5]);
    T.give(w[5]);
    T.give(-1);
    CHECK(T.others(-1) == 0);
    const int again = T.take();
    CHECK(again == w[5] && T.take() == -1);
    const uint32_t c = T.start(again);
    CHECK(T.others(w[0]) == 1);
    ended[again] = c;
    CHECK(T.others(w[0]) == 0);
    // many short-lived owners
    for (int r = 0; r < 10 * kFlightWords; ++r) {
        T.give(w[r % kFlightWords]);
        CHECK((w[r % kFlightWords] = T.take()) >= 0);
    }
    std::printf("flight words: ok\n");
    return 0;
}
