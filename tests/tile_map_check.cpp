// Check of the tile map (csrc/q38m_tiles.h) over row and column tile counts,
// for each of its orders: every tile belongs to exactly one workgroup of the
// grid; the XCDs' shares differ by at most one tile where columns are dealt or
// the rest is spread, and by at most one row tile otherwise; with rows dealt,
// a row tile of a whole group of eight stays on its XCD.  The chosen order
// never leaves an XCD without work where there are eight tiles.  Then the size
// limit: a grid that fits holds less than 2^32 threads, and its last
// workgroups lie inside the product.
//
// Prints the number of maps walked; exits with 1 and the first that fails.
#include "q38m_tiles.h"

#include <cstdio>
#include <vector>

using namespace q38m;

struct Shares {
    uint64_t least, most;
};

static bool walk(TileOrder order, uint32_t rows, uint32_t columns, Shares* shares) {
    const uint64_t grid = tile_grid(order, rows, columns);
    const uint64_t tiles = static_cast<uint64_t>(rows) * columns;
    if (grid % kTileXcds != 0u || grid < tiles) return false;
    std::vector<uint32_t> xcd_of(tiles, kTileXcds);
    uint64_t share[kTileXcds] = {};
    for (uint64_t w = 0; w < grid; ++w) {
        const TileAt at = tile_at(static_cast<uint32_t>(w), order, rows, columns);
        if (at.row >= rows) continue;
        if (at.column >= columns) return false;
        uint32_t& xcd = xcd_of[static_cast<uint64_t>(at.row) * columns + at.column];
        if (xcd != kTileXcds) return false;
        xcd = static_cast<uint32_t>(w % kTileXcds);
        ++share[xcd];
    }
    for (uint64_t t = 0; t < tiles; ++t) {
        if (xcd_of[t] == kTileXcds) return false;
        const uint64_t row = t / columns;
        if (order != kColumnTiles && row < rows / kTileXcds * kTileXcds && xcd_of[t] != row % kTileXcds)
            return false;
    }
    *shares = Shares{share[0], share[0]};
    for (uint64_t s : share) {
        shares->least = s < shares->least ? s : shares->least;
        shares->most = s > shares->most ? s : shares->most;
    }
    return shares->most - shares->least <= (order == kRowTiles ? columns : 1u);
}

int main() {
    unsigned maps = 0;
    const uint32_t some[] = {1u, 2u, 3u, 5u, 7u, 8u, 9u, 16u, 17u, 33u, 128u, 191u, 1187u};
    for (uint32_t a = 1; a <= 80u; ++a)
        for (uint32_t b : some)
            for (int swap = 0; swap < 2; ++swap) {
                const uint32_t rows = swap ? b : a, columns = swap ? a : b;
                Shares shares[3];
                for (TileOrder order : {kRowTiles, kRowTilesEven, kColumnTiles}) {
                    ++maps;
                    if (!walk(order, rows, columns, &shares[order])) {
                        std::printf("order %u rows %u columns %u\n", order, rows, columns);
                        return 1;
                    }
                }
                for (uint32_t k : {320u, 2048u})
                    for (uint64_t bytes : {uint64_t{0}, kInnerBytes}) {
                        const Shares& s = shares[tile_order(rows, columns, bytes, k)];
                        // (seven row tiles of few columns leave one XCD idle)
                        if (rows != 7u && static_cast<uint64_t>(rows) * columns >= 8u && s.least == 0u) {
                            std::printf("idle XCD: rows %u columns %u\n", rows, columns);
                            return 1;
                        }
                    }
            }
    // from one row tile to a square of them, the widest product that fits and
    // the next; 2^32 columns of 64
    struct Limit {
        TileOrder order;
        uint32_t rows, columns;
        bool fits;
    };
    for (const Limit& l :
         {Limit{kRowTilesEven, 1u, (1u << 24) - 8u, true}, Limit{kRowTilesEven, 1u, 1u << 24, false},
          Limit{kColumnTiles, 1u, (1u << 24) - 8u, true}, Limit{kColumnTiles, 1u, (1u << 24) - 7u, false},
          Limit{kRowTiles, 1u, (1u << 21) - 1u, true}, Limit{kRowTiles, 1u, 1u << 21, false},
          Limit{kRowTilesEven, 9u, 1864134u, true}, Limit{kRowTilesEven, 9u, 1864136u, false},
          Limit{kColumnTiles, 40u, 419430u, true}, Limit{kColumnTiles, 40u, 419431u, false},
          Limit{kRowTiles, 1u << 12, (1u << 12) - 1u, true}, Limit{kRowTiles, 1u << 12, 1u << 12, false},
          Limit{kColumnTiles, 1u << 15, 1u << 26, false}}) {
        const uint64_t grid = tile_grid(l.order, l.rows, l.columns);
        if (tile_grid_fits(l.order, l.rows, l.columns) != l.fits ||
            l.fits != (grid * 256u <= 0xffffffffull)) {
            std::printf("limit %u x %u: %llu\n", l.rows, l.columns, static_cast<unsigned long long>(grid));
            return 1;
        }
        for (uint64_t w = grid - 8u; l.fits && w < grid; ++w) {
            const TileAt at = tile_at(static_cast<uint32_t>(w), l.order, l.rows, l.columns);
            if (at.row < l.rows && at.column >= l.columns) {
                std::printf("last %u x %u\n", l.rows, l.columns);
                return 1;
            }
        }
    }
    std::printf("maps %u\n", maps);
    return 0;
}
