// The order in which workgroups take the tiles_m x tiles_n output tiles of a product, whose K may be in parts.
//
// Consecutive workgroups go to the eight XCDs in turn, each with an L2 of its own, so an XCD takes a run of neighbouring tiles (of the parts one after the
// other): panels of `panel` tile rows, column by column.  What its 32 CUs work on at a time then comes from `panel` activation slices and
// 32 / panel weight tiles, each read once into that L2.  A weight's bytes count twice, since the activations, which every XCD
// reads, come from the last-level cache and the weight from memory: time is least near panel^2 = 64 (weight tile) / (activation
// slice), with the tile rows dealt out evenly over that many panels.  Row by row (panel 1, all of one activation slice
// first) the weight came once per tile row; measured us, row by row / in panels: int8 14336 x 4096 at 190 / 450 / 1149 rows
// 35.4 / 34.0, 64.4 / 62.2, 138 / 134, 4096 x 14336 at 300 rows 57.6 / 51.2; FP6 14336 x 4096 at 80 / 450 rows 23.6 / 22.9, 63.9 / 60.6;
// int4 5120 x 13824 at 427 rows 102.3 / 96.2 (counting the weight once 102.0).  All rows in one panel is too much for many short rows (int4 1024 x
// 4096 at 2750 rows, 29 tile rows: 34.6 / 36.6).  The 256-row int4 tiles choose their own panels (int4wo_gemm.hip).
#pragma once
#include "common.h"
#include <math.h>

namespace ao {

struct TileOrder {
    int tiles_m, tiles_n, panel, parts;
    __host__ __device__ unsigned workgroups() const { return (unsigned)tiles_m * (unsigned)tiles_n * (unsigned)parts; }
};

// The item of `all` that workgroup `block` takes: each XCD a run of them, all runs of one length or of two that differ by one, and no workgroup without an item.
// (Runs of one length and a short last one, per part, had workgroups that ended at once: they still took a CU's turn, so that of the 41 tiles in six parts
// of int8 5128 x 13824 at 40 rows some CUs had two and others none, 37.2 us against 26.3; and the 33 tiles in seven parts of 4104 x 14336 gave the first XCDs 35 workgroups for
// 32 CUs, at 12 rows 32.0 us against 23.7.  In four parts of 4104 x 14336 at 96 rows 39.0 -> 27.2.)
__device__ __forceinline__ int xcd_run(int block, int all) {
    const int xcd = block & 7, even = all >> 3, more = all & 7;
    return xcd * even + (xcd < more ? xcd : more) + (block >> 3);
}

// x_bytes, w_bytes: what a tile reads of the activations and of the weight for the same stretch of K
inline TileOrder tile_order(int64_t tiles_m, int64_t tiles_n, int64_t x_bytes, int64_t w_bytes) {
    const int64_t per_xcd = (tiles_m * tiles_n + 7) / 8, at_once = per_xcd < 32 ? per_xcd : 32;
    const double high = sqrt(2.0 * (double)at_once * (double)w_bytes / (double)x_bytes);
    int64_t panels = high >= 1.0 ? (int64_t)((double)tiles_m / high + 0.5) : tiles_m;
    panels = panels < 1 ? 1 : panels;
    return TileOrder{(int)tiles_m, (int)tiles_n, (int)((tiles_m + panels - 1) / panels), 1};
}

// The tile of workgroup `block`, and its part of K
__device__ __forceinline__ void tile_at(const TileOrder& o, int block, int& tile_m, int& tile_n, int& part) {
    const int tiles = o.tiles_m * o.tiles_n;
    int tile = xcd_run(block, tiles * o.parts);
    // at most eight parts: compared rather than divided, since a division of scalars runs on the vector unit and leaves its result there
    part = 0;
#pragma unroll
    for (int z = 1; z < 8; ++z) part += tile >= z * tiles;
    part = __builtin_amdgcn_readfirstlane(part);
    tile -= part * tiles;
    const int per_panel = o.panel * o.tiles_n;
    int p = 0, in = tile;
    if (tile >= per_panel) p = tile / per_panel, in = tile - p * per_panel;
    const int high = min(o.panel, o.tiles_m - p * o.panel);
    tile_n = in / high;
    tile_m = p * o.panel + in - tile_n * high;
}

}  // namespace ao
