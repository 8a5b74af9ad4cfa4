// tpm_tile_order.hpp -- the order of one box's cells in the tile list, and
// back (no HIP dependency: also compiled for the host).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define TPM_HD __host__ __device__ __forceinline__
#else
#define TPM_HD inline
#endif

// Tile order: cells are visited in z-major blocks of TILE_BLOCK^3 cells
// (blocks z-major, cells z-major inside a block), so the tiles the PP kernel
// runs close together in time share their 27-cell neighbourhoods: a block's
// sources (10^3 cells at 512^3, ~2 MB) and its stretch of the potential mesh
// fit one XCD's L2.  rank(c) is this order's position of cell c, a bijection
// onto [0, C^3) (edge blocks are smaller).  Each tile is computed
// independently, so the order changes no result.
#define TILE_BLOCK 8
TPM_HD int32_t tile_min(int32_t a, int32_t b) { return a < b ? a : b; }
// 32-bit arithmetic throughout (C^3 < 2^27): a wave does this for one cell.
TPM_HD int32_t tile_rank(uint32_t c, uint32_t C) {
    const uint32_t q = c / C;
    const int x = (int)(c - q * C), z = (int)(q / C), y = (int)(q - (uint32_t)z * C), Ci = (int)C;
    const int bx = x / TILE_BLOCK, by = y / TILE_BLOCK, bz = z / TILE_BLOCK;
    const int sy = tile_min(TILE_BLOCK, Ci - by * TILE_BLOCK), sz = tile_min(TILE_BLOCK, Ci - bz * TILE_BLOCK);
    const int sx = tile_min(TILE_BLOCK, Ci - bx * TILE_BLOCK);
    const int before = bz * TILE_BLOCK * Ci * Ci + sz * by * TILE_BLOCK * Ci + sz * sy * bx * TILE_BLOCK;
    const int local = ((z - bz * TILE_BLOCK) * sy + (y - by * TILE_BLOCK)) * sx + (x - bx * TILE_BLOCK);
    return before + local;
}
// The cell whose rank is r.
TPM_HD int32_t tile_cell(uint32_t r, uint32_t C) {
    const int Ci = (int)C;
    int left = (int)r;
    const int bz = left / (TILE_BLOCK * Ci * Ci), sz = tile_min(TILE_BLOCK, Ci - bz * TILE_BLOCK);
    left -= bz * TILE_BLOCK * Ci * Ci;
    const int by = left / (sz * TILE_BLOCK * Ci), sy = tile_min(TILE_BLOCK, Ci - by * TILE_BLOCK);
    left -= by * sz * TILE_BLOCK * Ci;
    const int bx = left / (sz * sy * TILE_BLOCK), sx = tile_min(TILE_BLOCK, Ci - bx * TILE_BLOCK);
    left -= bx * sz * sy * TILE_BLOCK;
    const int q = left / sx, x = left - q * sx, z = q / sy, y = q - z * sy;
    return ((bz * TILE_BLOCK + z) * Ci + by * TILE_BLOCK + y) * Ci + bx * TILE_BLOCK + x;
}

// The chunk of tiles that slot v of the tile list finds: slots are spaced
// `space` tiles, a cell's chunks begin every ct >= space tiles from its first
// tile (first, of cell [first, end)).  Each chunk but a cell's first one or
// those a slot boundary coincides with is found by exactly one slot, that of
// the range [v space, (v + 1) space) that holds its first tile, when the cell
// is the one that holds tile v space.  Returns the chunk's number, or -1.
TPM_HD int32_t tile_slot_chunk(int64_t v, int32_t space, int32_t ct, int32_t first, int32_t end) {
    const int64_t s = v * space;
    const int64_t k = (s - first + ct - 1) / ct, t = first + k * ct;
    return t < end && t < s + space ? (int32_t)k : -1;
}
