// gps_list_growth.h — when a batch's point list is replaced by a longer one.
// The device falls back to the point-parallel splat when a list is too short,
// so a batch renders with whatever list there is.
#pragma once

#include <algorithm>
#include <cstdint>

namespace gps {

struct ListGrowth {
    uint64_t cap = 0;         // points of the list in use (0: none)
    uint64_t refused = ~0ull; // nothing as large as this is asked for again
    // Room for `points`, or as near to it as can be had: a list that is too
    // short is replaced by one of `preferred` points or twice its length where
    // that is more, else by one of exactly `points`.  alloc(n) replaces the
    // list and returns whether it could; without `may_alloc` it is not called.
    // False when there is no list at all.
    template <typename Alloc> bool reserve(uint64_t points, uint64_t preferred, bool may_alloc, Alloc alloc) {
        if (points > cap && may_alloc)
            for (uint64_t n : {std::max({points, preferred, 2 * cap}), points}) {
                if (n >= refused) continue;
                if (alloc(n)) {
                    cap = n;
                    break;
                }
                refused = n;
            }
        return cap != 0;
    }
};

}  // namespace gps
