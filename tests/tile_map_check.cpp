// Check of the tile map (csrc/q38m_tiles.h) over row and column tile counts:
// every tile belongs to exactly one workgroup of the grid, and a row tile
// stays on its XCD.  Then the size limit: a grid that fits holds less than
// 2^32 threads, and its last workgroups lie inside the product.
//
// Prints the number of maps walked; exits with 1 and the first that fails.
#include "q38m_tiles.h"

#include <cstdio>
#include <vector>

using namespace q38m;

static bool walk(uint32_t rows, uint32_t columns) {
    const uint64_t grid = tile_grid(rows, columns);
    const uint64_t tiles = static_cast<uint64_t>(rows) * columns;
    if (grid % kTileXcds != 0u || grid < tiles) return false;
    std::vector<uint32_t> xcd_of(tiles, kTileXcds);
    for (uint64_t w = 0; w < grid; ++w) {
        const TileAt at = tile_at(static_cast<uint32_t>(w), columns);
        if (at.row >= rows) continue;
        if (at.column >= columns) return false;
        uint32_t& xcd = xcd_of[static_cast<uint64_t>(at.row) * columns + at.column];
        if (xcd != kTileXcds) return false;
        xcd = static_cast<uint32_t>(w % kTileXcds);
    }
    for (uint64_t t = 0; t < tiles; ++t)
        if (xcd_of[t] != t / columns % kTileXcds) return false;
    return true;
}

int main() {
    unsigned maps = 0;
    for (uint32_t rows = 1; rows <= 80u; ++rows)
        for (uint32_t columns : {1u, 2u, 3u, 5u, 7u, 8u, 9u, 16u, 17u, 33u, 128u, 191u, 1187u}) {
            if (!walk(rows, columns)) {
                std::printf("rows %u columns %u\n", rows, columns);
                return 1;
            }
            ++maps;
        }
    // from one row tile to a square of them, the widest product that fits and
    // the next; 2^32 columns of 64
    struct Limit {
        uint32_t rows, columns;
        bool fits;
    };
    for (const Limit& l : {Limit{1u, (1u << 21) - 1u, true}, Limit{1u, 1u << 21, false},
                           Limit{1u, 1u << 23, false}, Limit{7u, (1u << 21) - 1u, true},
                           Limit{9u, (1u << 20) - 1u, true}, Limit{9u, 1u << 20, false},
                           Limit{1u << 12, (1u << 12) - 1u, true}, Limit{1u << 12, 1u << 12, false},
                           Limit{1u << 15, 1u << 26, false}}) {
        const uint64_t grid = tile_grid(l.rows, l.columns);
        if (tile_grid_fits(l.rows, l.columns) != l.fits || l.fits != (grid * 256u <= 0xffffffffull)) {
            std::printf("limit %u x %u: %llu\n", l.rows, l.columns, static_cast<unsigned long long>(grid));
            return 1;
        }
        for (uint64_t w = grid - 8u; l.fits && w < grid; ++w) {
            const TileAt at = tile_at(static_cast<uint32_t>(w), l.columns);
            if (at.row < l.rows && at.column >= l.columns) {
                std::printf("last %u x %u\n", l.rows, l.columns);
                return 1;
            }
        }
    }
    std::printf("maps %u\n", maps);
    return 0;
}
