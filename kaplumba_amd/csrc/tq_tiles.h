// 128-row tiles of the rotation kernels (tq_rotate.hip) in 32-bit row numbers.
// No HIP types: a host program includes it too (tests/csrc/tile_walk.cpp).
#pragma once

#include <cstdint>

namespace tq {

constexpr int kTileRows128 = 128;

// Most rows whose tiles number their rows in an int, the rows past the end of
// the last tile included (kernels clamp those).  Larger calls take the kernels
// with 64-bit indices.
constexpr int kMaxTiledRows = INT32_MAX - (kTileRows128 - 1);

constexpr int tiles_of(int rows) { return (rows + (kTileRows128 - 1)) / kTileRows128; }

static_assert(static_cast<int64_t>(tiles_of(kMaxTiledRows)) * kTileRows128 - 1 <= INT32_MAX, "last row of the last tile");
static_assert(static_cast<int64_t>(kMaxTiledRows) + (kTileRows128 - 1) <= INT32_MAX, "rows rounded up to whole tiles");

// A persistent workgroup's walk over tiles: counting tiles keeps the step past
// the last one (up to a grid of tiles) far from the int's end, where counting
// rows wrapped around.
template <typename F>
#ifdef __HIPCC__
__device__ __forceinline__
#else
inline
#endif
void walk_tiles(int rows, int first, int step, F f) {
  for (int t = first; t < tiles_of(rows); t += step) f(t * kTileRows128);
}

}  // namespace tq
