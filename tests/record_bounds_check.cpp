// The 16-bit bounds of a splat record (gps_project.h pack_bounds_min/max,
// packed_rect and packed_tiles, the source the GPU kernels compile) on the
// CPU: for every pair of tile edges near 0, the middle and the end of frames
// up to the largest, in each position of the packed word, the rectangle must
// hold exactly the pixels of [min, max) that lie below 65535, and the tiles
// exactly [min / 16, max / 16).  Prints the number of mismatches.
#include <cstdio>
#include <vector>

#include "gps_project.h"

using namespace gps;

int main() {
    const int sizes[] = {1, 16, 17, 1920, 65504, 65519, 65520, 65521, 65534, 65535};
    long bad = 0, checked = 0;
    auto edges = [](int size) {
        const int tiles = (size + 15) / 16;
        std::vector<int> e;
        for (int t : {0, 1, 2, tiles / 2, tiles - 2, tiles - 1, tiles})
            if (t >= 0 && t <= tiles) e.push_back(t * 16);
        return e;
    };
    for (int w : sizes)
        for (int h : sizes) {
            const std::vector<int> ex = edges(w), ey = edges(h);
            for (int x0 : ex)
                for (int x1 : ex)
                    for (int y0 : ey)
                        for (int y1 : ey) {
                            if (x1 < x0 || y1 < y0 || x0 >= w || y0 >= h) continue;  // as project_gaussian leaves them
                            Projected p{};
                            p.minx = x0, p.miny = y0, p.maxx = x1, p.maxy = y1;
                            const SampleRect r = packed_rect(pack_bounds_min(p), pack_bounds_max(p));
                            const TileRect t = packed_tiles(pack_bounds_min(p), pack_bounds_max(p));
                            const int ex1 = x1 < 65535 ? x1 : 65535, ey1 = y1 < 65535 ? y1 : 65535;
                            ++checked;
                            if (r.x0 != x0 || r.y0 != y0 || r.w != (uint32_t)(ex1 - x0) || r.h != (uint32_t)(ey1 - y0) ||
                                t.x0 != x0 / 16 || t.y0 != y0 / 16 || t.x1 != x1 / 16 || t.y1 != y1 / 16) {
                                if (bad < 5)
                                    std::printf("bounds [%d, %d) x [%d, %d): rect %d %d %u %u tiles %d %d %d %d\n", x0, x1,
                                                y0, y1, r.x0, r.y0, r.w, r.h, t.x0, t.y0, t.x1, t.y1);
                                ++bad;
                            }
                        }
        }
    std::printf("checked %ld mismatches %ld\n", checked, bad);
    return 0;
}
