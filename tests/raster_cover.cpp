// Every macro tile is taken exactly once, whatever the grid: by the workgroups, by the order that the hint
// reports, and where the tiles behind a wave are split over K and counted by position.
#include <cstdio>
#include <vector>

#include "fo_raster.h"

using namespace fo;

static bool once(const std::vector<int>& seen) {
    for (int n : seen)
        if (n != 1) return false;
    return true;
}

template <int GROUP, int UNIT>
static bool covers(int GM, int GN) {
    const unsigned magic = raster_magic(GN);
    const int total = GM * GN;
    const auto at = [&](TileCoord c) { return c.m >= 0 && c.m < GM && c.n >= 0 && c.n < GN ? c.m * GN + c.n : 0; };
    std::vector<int> mapped(total), order(total);
    for (int i = 0; i < total; ++i) {
        ++mapped[at(raster_map<GROUP, UNIT>(i, GM, GN, magic))];
        ++order[at(raster_order<GROUP, UNIT>(i, GM, GN, magic))];
    }
    if (!once(mapped) || !once(order)) return false;
    for (int from = 0; from <= total; from += kWave) {
        std::vector<int> split(total);
        for (int i = 0; i < total; ++i)
            ++split[at(i < from ? raster_map<GROUP, UNIT>(i, GM, GN, magic) : raster_tile<GROUP, UNIT>(i, GM, GN, magic, total))];
        if (!once(split)) return false;
    }
    return true;
}

int main() {
    for (int GM = 1; GM < 48; ++GM)
        for (int GN = 1; GN < 48; ++GN)
            if (!covers<8, 4>(GM, GN) || !covers<4, 8>(GM, GN)) {
                std::printf("%d x %d tiles are not covered once\n", GM, GN);
                return 1;
            }
    return 0;
}
