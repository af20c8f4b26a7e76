// gps_big.h — the list of the Gaussians that the binned splat leaves to global
// atomics, and how it stays in bounds.  A frame's points are 32-bit sums: where
// the total passes 2^32 the offsets wrap (as a sequential 32-bit scan's do), and
// the points below the budget are handed out once per turn, so a list sized by
// Gaussians and budget is too short.  Shared with the CPU test of these bounds.
#pragma once

#include "gps_detmath.h"

#define GPS_BIG_SLICE 1024u      // points that one workgroup takes at a time
#define GPS_BIG_ALL 0xFFFFFFFFu  // an item's start: all points of its Gaussian

namespace gps {

// The items of one such Gaussian of `points` points: its first slice has an item
// of its own (one per Gaussian, so there are no more than Gaussians), the other
// (points - 1) / GPS_BIG_SLICE are taken from `cap` shared ones, enough for the
// point budget (budget / GPS_BIG_SLICE).  big_rest: how many to take; the shared
// items counted so far say where they begin (`at`).
GPS_HD uint32_t big_rest(uint32_t points, uint32_t cap) {
    const uint32_t rest = (points - 1u) / GPS_BIG_SLICE;
    return rest < cap ? rest : cap;
}
// Stores the shared items with put(i, start) as far as there are any.  Returns
// the first item's start: 0, or GPS_BIG_ALL when the shared ones ran out, and
// the first item then stands for all of the points (some of them twice: a
// minimum does not mind).
template <typename Put>
GPS_HD uint32_t big_items(uint32_t points, uint32_t rest, uint32_t at, uint32_t cap, Put put) {
    const uint32_t room = at < cap ? cap - at : 0u;
    for (uint32_t j = 0; j < rest && j < room; ++j) put(at + j, (j + 1u) * GPS_BIG_SLICE);
    return rest <= room && rest == (points - 1u) / GPS_BIG_SLICE ? 0u : GPS_BIG_ALL;
}
// Points [lo, hi) of an item that starts at `start`, of a Gaussian of `points`.
GPS_HD uint32_t big_lo(uint32_t start) { return start == GPS_BIG_ALL ? 0u : start; }
GPS_HD uint32_t big_hi(uint32_t start, uint32_t points) {
    return start == GPS_BIG_ALL || points - start <= GPS_BIG_SLICE || points < start ? points : start + GPS_BIG_SLICE;
}

}  // namespace gps
