// gps_big.h — how the distributor counts points for the binned splat where a
// frame's point total passes 2^32.  The total and the offsets are 32-bit sums
// and wrap there (as a sequential 32-bit scan does), so points below the
// budget are then handed out once per turn: what is bounded by the budget in
// every other frame is not.  Shared with the CPU test of these bounds.
#pragma once

#include "gps_detmath.h"

#define GPS_BIG_SLICE 1024u         // points of a Gaussian too large to bin that one workgroup takes at a time
#define GPS_BIG_ALL 0xFFFFFFFFu     // an item's start: all points of its Gaussian

namespace gps {

// The items of one Gaussian too large to bin.  Its first slice has an item of
// its own (one per Gaussian, so there are no more than Gaussians); further
// slices are taken from `cap` shared items, enough for the point budget
// (budget / GPS_BIG_SLICE: a Gaussian of n points needs (n - 1) / GPS_BIG_SLICE).
// reserve(n) returns where n shared items begin, put(i, start) stores shared
// item i.  Returns the first item's start: 0, or GPS_BIG_ALL when the shared
// ones ran out, and the first item then stands for all of the points (some of
// them twice: a minimum does not mind).
template <typename Reserve, typename Put>
GPS_HD uint32_t big_items(uint32_t points, uint32_t cap, Reserve reserve, Put put) {
    const uint32_t rest = (points - 1u) / GPS_BIG_SLICE;
    if (rest == 0u) return 0u;
    const uint32_t at = rest <= cap ? reserve(rest) : cap;
    const uint32_t room = at < cap ? cap - at : 0u;
    for (uint32_t j = 0; j < rest && j < room; ++j) put(at + j, (j + 1u) * GPS_BIG_SLICE);
    return rest <= room ? 0u : GPS_BIG_ALL;
}
// Points [lo, hi) of an item that starts at `start`, of a Gaussian of `points`.
GPS_HD uint32_t big_lo(uint32_t start) { return start == GPS_BIG_ALL ? 0u : start; }
GPS_HD uint32_t big_hi(uint32_t start, uint32_t points) {
    return start == GPS_BIG_ALL || points - start <= GPS_BIG_SLICE || points < start ? points : start + GPS_BIG_SLICE;
}

// A tile's points per region are 32-bit sums in LDS.  Its 4096 Gaussians' points
// in units of 8192, rounded down, tell whether they can wrap: below 2^18 units
// there are fewer than 2^31 + 2^25 points, from there on 2^31, more than any
// list holds.
GPS_HD uint32_t point_units(uint32_t points) { return points >> 13; }
GPS_HD bool tile_too_large(uint32_t units) { return units >= 1u << 18; }

}  // namespace gps
