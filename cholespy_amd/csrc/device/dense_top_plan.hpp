// Lists for the dense top blocks of a plan (host side): the panels of the two
// products with X = L_TT^{-1} (dense_top.hip) and the tile products that form
// X (block_inverse.hip).
//
// X_ij is nonzero only where row i is an ancestor of row j (or j itself) in
// the elimination tree, so X is stored in the 16 x 16 units that hold such a
// pair: 2,122 units of 16,290 for a 61 x 47 grid, 9,076 of 23,871 for the top
// of icosphere(6), 55,732 of 76,636 for that of a 48^3 grid.
#pragma once
#include <cstdint>
#include <vector>

#include "block_plan.hpp"

namespace cholespy_amd {

constexpr int kTopUnit = 16;                          // rows and columns of a unit
constexpr int kTopUnitEntries = kTopUnit * kTopUnit;
constexpr int kTopTile = 64;                          // rows and columns of a tile of X while it is formed
constexpr int kTopTileEntries = kTopTile * kTopTile;

// Panels of more units than this are split among several workgroups: one
// streams 20 to 30 KB a microsecond, and the panels near the root have every
// row of the top as input. First product, whole panels against segments:
// icosphere(6), k = 16, FP64 (330 units) 27.3 -> 13.9 us, k = 128, FP32 43.0 ->
// 28.1, 33^3 grid, k = 5, FP64 24.9 -> 18.6, icosphere(7), k = 3, FP32 16.4 ->
// 13.0. (Twice the wavefronts a workgroup instead: 28.1, 42.0, 26.7.)
constexpr int kTopSegment = 96;

// One panel of 16 outputs of a product, or one of its segments: count input
// units from unit `first` on (w = X r: consecutive units of 16 rows), or those
// listed from position `first` of TopLists::units on (z = X' w). Segment `seg`
// of nseg leaves its sums in slot + seg of the segment sums; the last one to
// finish adds them up in order. Device record.
struct DenseTopPanel {
    int row0, n;      // first row of the top block and its rows
    int panel, sys;
    int first, count;
    int seg, nseg, slot, reserved;
    int64_t off;      // first element in the direction's array
};

struct TopLists {
    std::vector<DenseTopPanel> fwd, bwd;   // longest first: the last workgroups to start are the short ones
    std::vector<int> units;
    int slots = 0;                         // segment sums (the more of the two directions)
    int64_t entries = 0;                   // elements of one direction's array

    // Forming X. A block is a square of 64 x 64 tiles, of which those with an
    // ancestor pair exist; tile t is the kTopTileEntries column-major values
    // at t. They start as L and become X in place: the diagonal tiles are
    // inverted, then inverses of doubled size, X_21 = -X_22 (L_21 X_11), in
    // stages of independent jobs: into temporary tiles (L_21 X_11), then back.
    struct Column {
        int c, row0, map;          // column c of the block from row0, its tile map at map
    };
    struct Diagonal {
        int tile, rows;
    };
    struct Job {
        int out, first, count;     // pairs [first, first + count); out: temporary tile (even stages) or tile (odd)
    };
    struct Pair {
        int a, b;                  // even: tile, tile; odd: tile, temporary tile
    };
    // Blocks in groups whose work arrays stay within a bound (a block alone may
    // pass it); tiles and temporaries are counted from zero in each.
    struct Group {
        int tiles = 0, temps = 0;
        int columns[2], diagonals[2];        // ranges of the lists below
        int64_t fwd_units[2], bwd_units[2];
        std::vector<int> stages;             // job ranges: stage s is [stages[s], stages[s + 1])
    };
    std::vector<Group> groups;
    std::vector<Column> columns;
    std::vector<int> map;          // per block: tiles across, then the tile of (i, j) at i * across + j, -1 = none
    std::vector<Diagonal> diagonals;
    std::vector<Job> jobs;
    std::vector<Pair> pairs;
    // Per unit of the fwd and then of the bwd array: tile * 16 + unit row in
    // it * 4 + unit column (-1: no such tile, zeros).
    std::vector<int> pack;
};

constexpr int64_t kTopWorkBytes = int64_t(4) << 30;

// blk_sys: the system of each block (null: one system). work_bytes: a group's bound.
TopLists top_lists(const BlockPlan &P, const std::vector<int> *blk_sys, int64_t work_bytes = kTopWorkBytes);

}  // namespace cholespy_amd
