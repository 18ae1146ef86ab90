// Host check of kaplumba_amd/csrc/tq_tiles.h: every workgroup of a grid walks
// its tiles of the largest row counts, signed overflow trapped by the build
// (-fsanitize=undefined), and together they visit every tile once.
#include <cstdio>
#include <vector>

#include "tq_tiles.h"

int main() {
  using namespace tq;
  for (int rows : {1, 127, 128, 129, 100000, kMaxTiledRows - 128, kMaxTiledRows - 1, kMaxTiledRows}) {
    const int tiles = tiles_of(rows);
    for (int grid : {1, 3, 512, 4096}) {
      if (grid > tiles) continue;
      std::vector<unsigned char> seen(static_cast<size_t>(tiles), 0);
      for (int w = 0; w < grid; ++w) {
        walk_tiles(rows, w, grid, [&](int r0) {
          // the kernels' row numbers: r0 + a row of the tile, clamped below rows
          const int last = r0 + kTileRows128 - 1;
          if (r0 < 0 || last < r0 || r0 >= rows) __builtin_trap();
          ++seen[static_cast<size_t>(r0 / kTileRows128)];
        });
      }
      for (unsigned char s : seen)
        if (s != 1) return 1;
    }
  }
  std::puts("ok");
  return 0;
}
