// Host check of the order in which logged spikes are returned (eden_amd/csrc/event_order.hpp):
// equal to sorting them, over few and many events, rows at both ends of a run and before it.
//
// Build: g++ -std=c++17 -O1 -fsanitize=address -I<repo> event_order_check.cpp; prints "ok <trials>".
#include <cstdio>
#include <cstdlib>
#include <random>

#include "eden_amd/csrc/event_order.hpp"

int main() {
    std::mt19937 rng(5);
    int trials = 0;
    for (int64_t rows : {1, 2, 40, 1000})
        for (int n : {0, 1, 9, 10, 11, 500})
            for (int64_t first : {(int64_t)0, (int64_t)-1, (int64_t)-3}) {
                std::vector<int64_t> ev;
                for (int i = 0; i < n; i++) {
                    const int64_t row = first + (int64_t)(rng() % (uint32_t)(rows - first));
                    ev.push_back(row * (1 << 24) + (int64_t)(rng() % (1u << 24)));
                }
                if (n > 0) ev[0] = first * (1 << 24) + 0xFFFFFF;
                if (n > 1) ev[1] = (rows - 1) * (1 << 24);
                std::vector<int64_t> want = ev;
                std::sort(want.begin(), want.end());
                edenhip::order_events(ev, rows);
                if (ev != want) {
                    std::printf("rows %lld events %d first row %lld: another order\n", (long long)rows, n, (long long)first);
                    return 1;
                }
                trials++;
            }
    std::printf("ok %d\n", trials);
    return 0;
}
