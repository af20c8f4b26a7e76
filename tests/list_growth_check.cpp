// A batch's list growth (gps_list_growth.h) against an allocator that gives
// out at most `room` points.  Reads commands from argv: points, or "c" +
// points for a call that may not allocate.  Prints, per call, the list's
// length, the sizes asked for and whether there is a list.
#include <cstdio>
#include <cstdlib>
#include <string>

#include "gps_list_growth.h"

int main(int argc, char** argv) {
    const uint64_t room = strtoull(argv[1], nullptr, 10), preferred = strtoull(argv[2], nullptr, 10);
    gps::ListGrowth g;
    for (int i = 3; i < argc; ++i) {
        const bool may = argv[i][0] != 'c';
        std::string asked;
        const bool ok = g.reserve(strtoull(argv[i] + (may ? 0 : 1), nullptr, 10), preferred, may, [&](uint64_t n) {
            asked += " " + std::to_string(n);
            return n <= room;
        });
        std::printf("%llu %d asked%s\n", (unsigned long long)g.cap, ok ? 1 : 0, asked.c_str());
    }
    return 0;
}
