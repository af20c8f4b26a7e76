// The bounds of the list of large Gaussians (gps_big.h, the source the GPU
// distributor compiles) on the CPU, as the distributor uses them: Gaussians
// get 32-bit offsets that wrap past 2^32, and the points of each that lie
// below the budget.
// no item may lie outside its range, every point of every Gaussian must be in an
// item, and each once while nothing wraps.
// argv: Gaussians, points each (at most), budget, seed.  Prints the number of
// Gaussians with points, the turns, the items' shortfall and the faults.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "gps_big.h"

using namespace gps;

int main(int, char** argv) {
    const uint32_t n = (uint32_t)strtoul(argv[1], nullptr, 10), most = (uint32_t)strtoul(argv[2], nullptr, 10);
    const uint32_t budget = (uint32_t)strtoul(argv[3], nullptr, 10);
    uint64_t x = strtoull(argv[4], nullptr, 10) * 0x9E3779B97F4A7C15ull + 1;
    const uint32_t cap = budget / GPS_BIG_SLICE + 1;
    struct Item {
        uint32_t r, start;
    };
    std::vector<Item> first, shared(cap, Item{0, 0});
    std::vector<uint8_t> written(cap, 0);
    std::vector<uint32_t> pts(n);
    uint64_t total = 0, faults = 0, all = 0, with = 0;
    uint32_t used = 0;
    std::vector<uint32_t> w(n);
    for (uint32_t r = 0; r < n; ++r) {
        x ^= x << 13, x ^= x >> 7, x ^= x << 17;
        w[r] = most > 1 ? most / 2 + (uint32_t)(x % (most - most / 2)) + 1 : 1;
        total += w[r];
    }
    const uint32_t p_end = (uint32_t)total < budget ? (uint32_t)total : budget;
    uint32_t o = 0;
    for (uint32_t r = 0; r < n; ++r) {
        const uint32_t hi = o + w[r] < p_end ? o + w[r] : p_end;
        pts[r] = o < hi ? hi - o : 0u;
        o += w[r];
        if (pts[r]) {
            ++with;
            const uint32_t rest = big_rest(pts[r], cap), at = used;
            used += rest;
            const uint32_t start = big_items(pts[r], rest, at, cap, [&](uint32_t i, uint32_t s) {
                if (i >= cap || written[i]) ++faults;
                else shared[i] = Item{r, s}, written[i] = 1;
            });
            first.push_back(Item{r, start});
            all += start == GPS_BIG_ALL;
        }
    }
    const uint32_t n2 = used < cap ? used : cap;
    std::vector<uint64_t> covered(n, 0);
    auto take = [&](const Item& it) {
        const uint32_t lo = big_lo(it.start), hi = big_hi(it.start, pts[it.r]);
        if (lo < hi) covered[it.r] += hi - lo;
    };
    for (const Item& it : first) take(it);
    for (uint32_t i = 0; i < n2; ++i) {
        if (!written[i]) ++faults;
        take(shared[i]);
    }
    for (uint32_t r = 0; r < n; ++r)
        if (covered[r] < pts[r] || (total < (1ull << 32) && covered[r] != pts[r])) ++faults;
    if (first.size() > n) ++faults;
    std::printf("with %llu turns %llu short %llu faults %llu\n", (unsigned long long)with,
                (unsigned long long)(total >> 32), (unsigned long long)all, (unsigned long long)faults);
    return 0;
}
