// Order of a tiled product's workgroups (csrc/gpu/tile_order.h): every tile is taken exactly once,
// and no XCD has many more tiles than its share: by columns at most ceil(col_tiles / 8)
// columns, which is what one order alone gave, and beyond 16 tiles never more than the other
// order's busiest XCD by more than an eighth.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../cgcl-coraanns_amd/csrc/gpu/tile_order.h"

int main() {
    for (uint32_t nr : {1u, 2u, 3u, 4u, 5u, 7u, 8u, 9u, 31u, 32u, 33u, 79u, 257u})
        for (uint32_t nc = 1; nc <= 70; ++nc) {
            const cora::TileOrder o = cora::tile_order(nr, nc);
            std::vector<int> taken(nr * nc, 0);
            uint32_t load[8] = {};
            for (uint32_t b = 0; b < o.blocks; ++b) {
                uint32_t r, c;
                cora::tile_of(b, o.cols, nc, r, c);
                if (r >= nr || c >= nc)
                    continue;
                ++taken[r * nc + c];
                ++load[b % 8];
            }
            const uint32_t busiest = *std::max_element(load, load + 8);
            const uint32_t by_cols = (nc + 7) / 8 * nr, by_rows = (nr + 7) / 8 * nc;
            const bool once = std::all_of(taken.begin(), taken.end(), [](int n) { return n == 1; });
            if (!once || busiest > by_cols || (busiest > 16 && 7 * busiest > 8 * by_rows)) {
                std::printf("FAIL %u x %u tiles: once %d busiest %u by columns %u by rows %u\n", nr, nc, (int)once,
                            busiest, by_cols, by_rows);
                return 1;
            }
        }
    std::printf("PASS\n");
    return 0;
}
