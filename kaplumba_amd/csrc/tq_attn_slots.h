// LDS slots of decoded key rows and value rows in the kernels that share one
// decoded 32-token tile among waves (tq_attn_tile.h, tq_attn_wide.h).
#pragma once

namespace tq {

// Slot of token t's decoded key row: row m = 4 (t / 8) + t % 4 of tile
// h = (t / 4) % 2, so that score lane group g collects tokens 8 g .. 8 g + 7.
__device__ __forceinline__ int tile_kslot(int t) { return 16 * ((t >> 2) & 1) + 4 * (t >> 3) + (t & 3); }

// Slot of token t's 32-byte row in a 16-column value block: bit 3 of t
// folded into bit 2, so the eight rows a half-wave's transposed read touches
// (8 g + 4 h + 0..3 for g = 2 k, 2 k + 1) sit in eight distinct 32-byte bank
// groups.  An involution, hence a permutation of 0..31.
__device__ __forceinline__ int tile_vslot(int t) { return t ^ ((t >> 1) & 4); }

}  // namespace tq
