// Which output tile each workgroup of a tiled product takes, on a chip of eight XCDs to which
// workgroups go in turn (block % 8) and which have an L2 each.
//
// By columns: XCD x owns column tiles [x cols, (x + 1) cols), swept by groups of four row tiles,
// so the workgroups resident on an XCD share their operand tiles in its L2. By rows (cols == 0):
// XCD x owns the row tiles x, x + 8, ..., in groups of four that sweep all column tiles, for
// products with too few column tiles for eight owners: with one of them (128 columns or
// fewer) an eighth of the chip would do the work. 12,288 rows of 256 against 256 columns: by
// columns 32.1 us, by rows 17.6.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define CORA_HOST_DEVICE __host__ __device__
#else
#define CORA_HOST_DEVICE
#endif

namespace cora {

struct TileOrder {
    uint32_t cols;    // column tiles an XCD owns, or 0: row tiles are owned
    uint32_t blocks;  // workgroups to launch (some find no tile)
};

// The order whose busiest XCD has fewer tiles; by columns unless rows save an eighth of them (the
// sweep by rows reads the column operand once per XCD and group), and while the busiest has at
// most 16 of them, for half its 32 CUs: nothing queues then (777 queries of 384 dimensions against
// 1,500 centroids, 14 tiles by columns and 12 by rows: 24.7 and 30.3 us).
inline TileOrder tile_order(uint32_t row_tiles, uint32_t col_tiles) {
    const uint32_t cols = (col_tiles + 7) / 8, rows = (row_tiles + 7) / 8;
    const uint64_t by_cols = (uint64_t)cols * row_tiles, by_rows = (uint64_t)rows * col_tiles;
    if (by_cols > 16 && 8 * by_rows < 7 * by_cols)
        return {0, 8 * 4 * col_tiles * ((rows + 3) / 4)};
    return {cols, 8 * 4 * cols * ((row_tiles + 3) / 4)};
}

// The tile of workgroup `block`; the workgroup has none where row >= row_tiles or col >= col_tiles.
CORA_HOST_DEVICE inline void tile_of(uint32_t block, uint32_t cols, uint32_t col_tiles, uint32_t &row, uint32_t &col) {
    const uint32_t xcd = block % 8, i = block / 8;
    const uint32_t wide = 4 * (cols ? cols : col_tiles);  // tiles of a group of four row tiles
    const uint32_t group = i / wide, within = i % wide;
    row = 4 * group + within % 4;
    col = within / 4;
    if (cols)
        col += xcd * cols;
    else
        row = 8 * row + xcd;
}

}  // namespace cora
