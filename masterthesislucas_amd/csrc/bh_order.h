// Host side of bh_batch_order_by_cost: the work entries of a batched context by the cost of their
// last walk. Plain C++, also compiled by the tests.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cstddef>
#include <vector>

namespace bh {

// counts: two interaction counts per wave of the walk; entry[w]: the entry that wave w walked (an
// entry's slices add up); sinks(e): sinks of entry e. cost[e]: interactions per sink, since a wave's
// walk is shared by its lanes and its time does not follow their number. order: the entries in
// descending cost, ties by entry.
// A stable radix sort, 11 bits a pass over the bits of the largest cost, and the wave's entry at hand:
// the whole call takes 0.15 ms for 128 systems (1.95M particles, 30,600 entries). Sorting (cost,
// entry) pairs after a search for each wave's entry by its first sink took 2.3 (and 1.06 when an
// entry held 128 sinks).
template <typename Sinks>
inline void order_by_cost(const unsigned long long* counts, const uint32_t* entry, size_t waves,
                          size_t entries, Sinks sinks, std::vector<unsigned long long>& cost,
                          std::vector<uint32_t>& order) {
    constexpr int kBits = 11;
    constexpr size_t kBins = size_t(1) << kBits;
    cost.assign(entries, 0ull);
    for (size_t w = 0; w < waves; ++w) cost[entry[w]] += counts[2 * w] + counts[2 * w + 1];
    unsigned long long top = 0;
    for (size_t e = 0; e < entries; ++e) {
        const uint32_t s = sinks(e);
        cost[e] = s == 64 ? cost[e] >> 6 : s ? cost[e] / s : cost[e];
        top = std::max(top, cost[e]);
    }
    order.resize(entries);
    for (size_t e = 0; e < entries; ++e) order[e] = (uint32_t)e;
    std::vector<uint32_t> next(entries);
    std::vector<size_t> at(kBins);
    for (int shift = 0; shift < 64 && (top >> shift) != 0; shift += kBits) {
        const auto digit = [&](uint32_t e) { return ((top - cost[e]) >> shift) & (kBins - 1); };
        std::fill(at.begin(), at.end(), 0);
        for (size_t e = 0; e < entries; ++e) ++at[digit((uint32_t)e)];
        size_t sum = 0;
        for (size_t& a : at) {
            const size_t c = a;
            a = sum;
            sum += c;
        }
        for (uint32_t e : order) next[at[digit(e)]++] = e;
        order.swap(next);
    }
}

}  // namespace bh
