// tpm_tiles.hpp -- the direct kernel's work items (tpm_tiles.hip).
#pragma once

#include "tpm_internal.hpp"

// The cells of one box (boxes null: C, cell_w, min_rung and the cell box
// [lo, hi) apply) or of every live box of a batch.
struct tpm_tile_args {
    const uint32_t* x;
    const uint32_t* y;
    const uint32_t* z;
    const int8_t* rung;
    const int32_t* cell_begin;
    int32_t ncell;
    int32_t nbox;
    const tpm_box_dev* boxes;
    int C, min_rung;
    int64_t n;        // particles of the box (boxes: in the table)
    int64_t n_all;    // particles of all cells
    int per_cell;     // waves per cell of the build (this and the next two set by tpm_tiles_make)
    int group;        // cells per wave of the build, of which a lane makes those with one tile; 0: per_cell waves
    int slot_waves;   // waves that find the chunks of crowded cells
    uint32_t cell_w;
    int3 lo, hi;
    int ts;
    int all;          // tiles hold every particle, active or not
    int full;         // 1: every tile of a cell but its last has exactly ts sinks, 0: of even size
    int32_t* cnt;     // ncell: tiles per cell
    int32_t* off;     // ncell + 1: their exclusive scan, then the number of tiles
    int32_t* part;    // ncell / 2048 + 2: scan scratch
    int4* tiles;      // (cell, begin, end, box), ranges of order; nullptr: only the order is wanted
    uint32_t* order;  // particles, cell by cell
};

// The raw positions in the order of the tiles.
tpm_status tpm_order_positions(std::string& err, hipStream_t s, int64_t n, const tpm_tile_args& a, uint32_t* x,
                               uint32_t* y, uint32_t* z);
// Tiles of at most ts active sinks of one cell, in spatial order.
tpm_status tpm_tiles_make(std::string& err, hipStream_t s, tpm_tile_args a);
