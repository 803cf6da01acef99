// Tile map of the one-dimensional grids that cover row x column output tiles
// (the dense workgroup tiles and the hyper-connection mix-up).  Plain C++:
// the launches size their grids and the kernels find their tile by it, and
// a host program checks it (tests/tile_map_check.cpp).
//
// The dispatcher hands workgroups to the 8 XCDs round-robin by id, and each
// XCD has its own L2 of 4 MB.  Three orders:
// - kRowTiles: XCD x (workgroups x, x + 8, ...) runs row tiles x, x + 8, ...,
//   all column tiles of one before the next, so that a row tile's operand is
//   fetched into one L2; the row tiles past the last whole group of eight
//   are those of the first XCDs.
// - kRowTilesEven: the same, but that rest's tiles, row by row, are spread
//   over the XCDs in eight contiguous ranges (and come first).
// - kColumnTiles: all tiles, column by column, in eight contiguous ranges:
//   the column operand is fetched once, the row operand into every L2.
#pragma once

#include <stdint.h>

namespace q38m {

constexpr uint32_t kTileXcds = 8;

enum TileOrder : uint32_t { kRowTiles, kRowTilesEven, kColumnTiles };

// The order of a product whose B operand (`columns` tiles) is `column_bytes`
// long, over k values of K; both sides' tiles are equally large.
//
// Columns are dealt where there are more of them and B does not stay in an L2
// beside the row tiles that pass by: with rows dealt every XCD streams all of B
// again for each of its row tiles, and a product of one to seven row tiles
// leaves XCDs idle.  Above 40 row tiles the XCDs write too far apart.  Rows /
// columns dealt, us, 64 x 64 or 128 x 128 tiles: 2 x 65,536 x 2,048 223 / 40, 200
// x 16,384 x 2,048 73 / 29, 512 x 8,192 x 768 19.0 / 12.8, 3,000 x 8,192 x 320
// 32.4 / 24.8, 4,099 x 8,192 x 512 (33 row tiles) 60.1 / 50.4; 6,000 x 16,384 x
// 192 (47) 79.2 / 90.8, 8,192 x 16,384 x 512 (64) 215 / 303.  The line in B: 2.9 MB,
// 2,049 x 6,016 x 256 17.5 / 14.1, 3,000 x 3,000 x 512 15.9 / 16.5; 2.5 MB, 1,100 x
// 4,096 x 320 8.6 / 7.9; 2.2 MB, 1,400 x 6,016 x 192 9.2 / 9.7; 2.0 MB, 3,000 x 4,096
// x 256 13.0 / 13.9.
//
// With rows dealt the rest is spread where the first XCDs would hold a quarter
// more tiles than the mean: the mix-up of a single channel pair ran on one
// XCD (hidden 32, 6,500 tokens 39.5 -> 30.0 us), 600 tokens at hidden 2,048 45.0
// -> 41.5, a shared expert of inter 4,096 over 2,049 tokens 191 -> 174.  A spread
// tile's operand is fetched by another XCD, and a product's last writes leave
// all eight L2s at once, which short products do not earn back (1,537 x
// 2,048 x 512 7.5 -> 8.5, 2,049 x 4,096 x 192 9.7 -> 11.4): those spread up to seven
// row tiles, and up to twelve where two of them are more than the 64 128 x 128
// tiles an XCD holds at once (1,025 x 6,016 x 192, 9 x 47 tiles, 9.9 -> 7.6; 513 x
// 2,048 x 512, 9 x 32, 4.7 -> 5.3).
constexpr uint64_t kInnerBytes = 5u << 19;  // 2.5 MB
constexpr TileOrder tile_order(uint32_t rows, uint32_t columns, uint64_t column_bytes, uint32_t k) {
    if (columns > rows && rows <= 40u && column_bytes >= kInnerBytes) return kColumnTiles;
    const uint32_t groups = rows / kTileXcds, rest = rows % kTileXcds;
    const bool spread = rest != 0u && 8u * groups + 5u * rest <= 32u;
    const bool short_k = k <= 1024u && groups != 0u && (groups > 1u || columns <= 32u);
    return spread && !short_k ? kRowTilesEven : kRowTiles;
}

// workgroups that cover rows x columns tiles
constexpr uint64_t tile_grid(TileOrder order, uint32_t rows, uint32_t columns) {
    const uint64_t all = static_cast<uint64_t>(rows) * columns;
    const uint64_t whole = static_cast<uint64_t>(rows / kTileXcds) * columns;  // ids per XCD
    if (order == kColumnTiles) return (all + kTileXcds - 1u) / kTileXcds * kTileXcds;
    if (order == kRowTilesEven)
        return (whole + (all - whole * kTileXcds + kTileXcds - 1u) / kTileXcds) * kTileXcds;
    return static_cast<uint64_t>((rows + kTileXcds - 1u) / kTileXcds) * kTileXcds * columns;
}

// A grid dimension of 256-thread workgroups holds less than 2^32 threads.
constexpr bool tile_grid_fits(TileOrder order, uint32_t rows, uint32_t columns) {
    return tile_grid(order, rows, columns) < (1ull << 24);
}

struct TileAt {
    uint32_t row, column;  // row >= rows: no tile
};

constexpr TileAt tile_at(uint32_t workgroup, TileOrder order, uint32_t rows, uint32_t columns) {
    const uint32_t xcd = workgroup % kTileXcds;
    uint32_t j = workgroup / kTileXcds;
    if (order != kRowTiles) {
        const uint32_t spread = order == kColumnTiles ? rows : rows % kTileXcds;
        const uint32_t tiles = spread * columns;
        const uint32_t per = tiles / kTileXcds, extra = tiles % kTileXcds;
        const uint32_t ids = per + (extra != 0u ? 1u : 0u);  // of each XCD
        if (j < ids) {
            if (j == per && xcd >= extra) return TileAt{rows, 0u};
            const uint32_t tile = xcd * per + (xcd < extra ? xcd : extra) + j;
            return order == kColumnTiles ? TileAt{tile % rows, tile / rows}
                                         : TileAt{rows - spread + tile / columns, tile % columns};
        }
        j -= ids;
    }
    return TileAt{j / columns * kTileXcds + xcd, j % columns};
}

}  // namespace q38m
