// Tile map of the one-dimensional grids that cover row x column output tiles
// (the dense workgroup tiles and the hyper-connection mix-up).  Plain C++:
// the launches size their grids and the kernels find their tile by it, and
// a host program checks it (tests/tile_map_check.cpp).
//
// The dispatcher hands workgroups to the 8 XCDs round-robin by id, and each
// XCD has its own L2.  XCD x (workgroups x, x + 8, ...) runs row tiles x,
// x + 8, ..., all column tiles of one before the next, so that a row tile's
// operand is fetched into one L2.
#pragma once

#include <stdint.h>

namespace q38m {

constexpr uint32_t kTileXcds = 8;

// workgroups that cover rows x columns tiles
constexpr uint64_t tile_grid(uint32_t rows, uint32_t columns) {
    return static_cast<uint64_t>((rows + kTileXcds - 1u) / kTileXcds) * kTileXcds * columns;
}

// A grid dimension of 256-thread workgroups holds less than 2^32 threads.
constexpr bool tile_grid_fits(uint32_t rows, uint32_t columns) {
    return tile_grid(rows, columns) < (1ull << 24);
}

struct TileAt {
    uint32_t row, column;  // row >= rows: no tile
};

constexpr TileAt tile_at(uint32_t workgroup, uint32_t columns) {
    const uint32_t j = workgroup / kTileXcds;
    return TileAt{j / columns * kTileXcds + workgroup % kTileXcds, j % columns};
}

}  // namespace q38m
