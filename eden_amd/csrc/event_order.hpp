// event_order.hpp -- the order in which edenhip_read_events returns logged spikes. Host only.
#ifndef EDENHIP_EVENT_ORDER_HPP
#define EDENHIP_EVENT_ORDER_HPP

#include <algorithm>
#include <cstdint>
#include <vector>

namespace edenhip {

// Events (row << 24 | column) in ascending order: counted into rows, then the few events of each
// row sorted (many events), or sorted outright (few). A point neuron's generated step may raise a
// spike in the steps before row 0, whose row is negative: such events are sorted outright too, as
// the counters are indexed by row.
inline void order_events(std::vector<int64_t> &ev, int64_t total_rows) {
    bool counted = (int64_t)ev.size() * 4 > total_rows;
    for (size_t i = 0; i < ev.size() && counted; i++) {
        const int64_t r = ev[i] >> 24;
        counted = r >= 0 && r <= total_rows;
    }
    if (!counted) {
        std::sort(ev.begin(), ev.end());
        return;
    }
    std::vector<uint32_t> at((size_t)total_rows + 2, 0u);
    for (int64_t x : ev) at[(size_t)(x >> 24) + 1]++;
    for (size_t r = 1; r < at.size(); r++) at[r] += at[r - 1];
    std::vector<int64_t> by_row(ev.size());
    for (int64_t x : ev) by_row[at[(size_t)(x >> 24)]++] = x;
    ev.swap(by_row);
    for (size_t b = 0; b < ev.size();) {
        size_t e = b + 1;
        while (e < ev.size() && (ev[e] >> 24) == (ev[b] >> 24)) e++;
        std::sort(ev.begin() + (int64_t)b, ev.begin() + (int64_t)e);
        b = e;
    }
}

}  // namespace edenhip

#endif
