// csrc/bh_order.h against a sort of (cost, entry) pairs and a search for each wave's entry by its
// first sink, which is how the table was ordered before. Prints the milliseconds of both, the
// sorted form over half as many entries (it then had 128 sinks each, now 64).
#include <chrono>
#include <cstdio>
#include <random>
#include <utility>

#include "../masterthesislucas_amd/csrc/bh_order.h"

typedef unsigned long long u64;

struct Table {
    std::vector<u64> counts;                           // per wave, two
    std::vector<uint32_t> entry, first, sinks, wave1;  // per wave, per entry x 2, per wave
};

static Table make(size_t n, uint32_t per, int slices, u64 top, uint32_t seed) {
    std::mt19937_64 g(seed);
    Table t;
    uint32_t at = 0;
    for (size_t e = 0; e < n; ++e) {
        const uint32_t s = g() % 8 ? per : 1 + (uint32_t)(g() % per);
        t.first.push_back(at);
        t.sinks.push_back(s);
        at += s;
    }
    std::vector<uint32_t> place(n);
    for (size_t e = 0; e < n; ++e) place[e] = (uint32_t)e;
    std::shuffle(place.begin(), place.end(), g);  // a table that was ordered before
    for (size_t k = 0; k < n; ++k)
        for (int f = 0; f < (k < n / 50 ? slices : 1); ++f) {
            const u64 range = top >> (g() % 40), c = range ? g() % range : 0;
            t.entry.push_back(place[k]);
            t.wave1.push_back(t.first[place[k]]);
            t.counts.push_back(g() % 5 ? c : 1000);  // ties
            t.counts.push_back(g() % 5 ? c / 3 : 64);
        }
    return t;
}

static void by_sort(const Table& t, std::vector<u64>& cost, std::vector<uint32_t>& order) {
    const size_t n = t.first.size();
    std::vector<std::pair<uint32_t, uint32_t>> by_first(n);
    for (size_t i = 0; i < n; ++i) by_first[i] = {t.first[i], (uint32_t)i};
    std::sort(by_first.begin(), by_first.end());
    cost.assign(n, 0ull);
    for (size_t w = 0; w < t.entry.size(); ++w) {
        const auto it = std::lower_bound(by_first.begin(), by_first.end(),
                                         std::make_pair(t.wave1[w], 0u));
        cost[it->second] += t.counts[2 * w] + t.counts[2 * w + 1];
    }
    for (size_t i = 0; i < n; ++i) cost[i] /= t.sinks[i];
    std::vector<std::pair<u64, uint32_t>> ord(n);
    for (size_t i = 0; i < n; ++i) ord[i] = {~cost[i], (uint32_t)i};
    std::sort(ord.begin(), ord.end());
    order.resize(n);
    for (size_t i = 0; i < n; ++i) order[i] = ord[i].second;
}

template <typename F>
static double best_ms(F f) {
    double best = 1e30;
    for (int k = 0; k < 7; ++k) {
        const auto t0 = std::chrono::steady_clock::now();
        f();
        best = std::min(best, std::chrono::duration<double, std::milli>(
                                  std::chrono::steady_clock::now() - t0).count());
    }
    return best;
}

int main() {
    std::vector<u64> c0, c1;
    std::vector<uint32_t> o0, o1;
    for (size_t n : {1, 2, 63, 1000, 30000})
        for (u64 top : {0ull, 1ull, 2047ull, 2048ull, 1ull << 22, 1ull << 33, 1ull << 60}) {
            const Table t = make(n, 64, 8, top, (uint32_t)n + 7);
            by_sort(t, c0, o0);
            bh::order_by_cost(t.counts.data(), t.entry.data(), t.entry.size(), n,
                              [&](size_t e) { return t.sinks[e]; }, c1, o1);
            if (c0 != c1 || o0 != o1) {
                std::printf("FAIL n=%zu top=%llu\n", n, top);
                return 1;
            }
        }
    const size_t n = 40000;
    const Table now = make(n, 64, 8, 1ull << 26, 1), then = make(n / 2, 128, 8, 1ull << 26, 1);
    const double a = best_ms([&] { by_sort(then, c0, o0); });
    const double b = best_ms([&] {
        bh::order_by_cost(now.counts.data(), now.entry.data(), now.entry.size(), n,
                          [&](size_t e) { return now.sinks[e]; }, c1, o1);
    });
    std::printf("OK %.3f %.3f\n", a, b);
    return 0;
}
