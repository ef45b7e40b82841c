// The ring kernel's tile order: which tiles of a launch the blocks of an XCD compute, in which order.  Host and device code, so
// that a host program can walk every XCD's share.
#pragma once

#include <hip/hip_runtime.h>

namespace fmoe {

// Tiles are numbered in groups of GROUP_M row tiles x all column tiles.  Whole rounds of XCDS groups are dealt one group to
// every XCD, back and forth (in odd rounds XCD x takes position XCDS - 1 - x): rows shared by concurrent tiles meet in one L2,
// and no XCD is handed all the long experts, which come sorted by load often enough.
//
// What is left after the whole rounds goes out as groups as well, or as an equal run of tiles per XCD.  Dealt as groups, a launch
// of few groups keeps one XCD's blocks at work for a round or two while others are done (us per GEMM, groups / runs: 9189
// rows, 12 experts, 1024 -> 2560 columns 76.9 / 58.3; 16384 rows, 8 experts, 1024 -> 4096 176.6 / 151.5).  Runs share no operands
// between their XCDs, so they are taken where they shorten the launch:
//   * the busiest XCD is a round of tiles shorter (`slots` blocks each);
//   * one round holds even the busiest XCD's tiles: all run at once, and spread out they have every XCD's bandwidth (8509
//     rows, 12 experts, 2624 -> 1024 62.7 / 53.7; 4476 rows, 3136 -> 2048 74 / 67);
//   * its last round is three quarters full or more, and more than one group is left (20294 rows, 4 experts, 1792 -> 2560
//     178 / 169; with three quarters of a group left, 16384 rows, 8 experts, 4096 -> 2 x 1024, Zipf 265 / 274).
// Tiles of unequal cost (contraction windows, the longest first) go out in runs only where there is no whole round: after one,
// the left-over groups are the cheapest and belong to the XCDs that had the shorter windows (weight gradients of 9189 rows, 12
// experts, 1000 x 2600, Zipf 138 / 148; 2600 x 1000 75.7 / 77.2; one expert, 4096 x 4096, no whole round 462 / 232).
// Otherwise they only give every XCD a last round of its own: 6138 rows, 12 experts, 3648 -> 4096 (16 tiles left, 80 on one XCD
// or 66 on each, 32 slots) 209 / 234; 24576 rows, 64 experts, 2048 -> 1408 195 / 202.  Seven groups and more are as good as a round.
template <typename tile_t, int XCDS, int GROUP_M, bool EQUAL_COST = true>
struct TileDeal {
    tile_t span;        // tiles of a group
    tile_t count;       // tiles of this XCD
    tile_t dealt;       // of them in whole groups
    tile_t run_base;    // number of the run's first tile, less dealt
    int xcd;

    __host__ __device__ __forceinline__ TileDeal() {}
    __host__ __device__ __forceinline__ TileDeal(int row_tiles, int n_tiles, int xcd_, int slots) : xcd(xcd_) {
        span = (tile_t)GROUP_M * n_tiles;
        const int rounds = row_tiles / (GROUP_M * XCDS);
        const tile_t whole = rounds * span, rest = (tile_t)row_tiles * n_tiles - whole * XCDS;
        const tile_t even = (rest + XCDS - 1) / XCDS;
        const tile_t busiest = whole + (rest < span ? rest : span);
        const tile_t last_round = busiest > 0 ? (busiest - 1) % slots + 1 : 0;
        const bool runs = rest < (XCDS - 1) * span && (EQUAL_COST || rounds == 0) &&
                          (busiest <= slots || busiest - (whole + even) >= last_round || (4 * last_round >= 3 * slots && rest > span));
        const tile_t run = runs ? even : span;
        const int pos = runs || !(rounds & 1) ? xcd : XCDS - 1 - xcd;
        const tile_t left = rest - pos * run;
        count = whole + (left < 0 ? 0 : left < run ? left : run);
        dealt = runs ? whole : count;
        run_base = whole * (XCDS - 1) + pos * run;
    }

    // one contiguous range of the tile order per XCD
    static __host__ __device__ __forceinline__ TileDeal contiguous(int row_tiles, int n_tiles, int xcd) {
        TileDeal d;
        const tile_t total = (tile_t)row_tiles * n_tiles, share = (total + XCDS - 1) / XCDS;
        d.run_base = xcd * share;
        d.count = total - d.run_base < share ? total - d.run_base : share;      // (none: <= 0)
        d.span = d.dealt = 0;
        d.xcd = xcd;
        return d;
    }

    // number of this XCD's j-th tile; round = j / span
    __host__ __device__ __forceinline__ tile_t tile(tile_t j, tile_t round) const {
        if (j >= dealt) return run_base + j;
        const int pos = (round & 1) ? XCDS - 1 - xcd : xcd;
        return (round * XCDS + pos) * span + (j - round * span);
    }
};

}  // namespace fmoe
