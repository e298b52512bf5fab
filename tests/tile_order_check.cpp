// Host check of the tile order of a terrain's cells (tile_map, tile_index,
// tile_xy in simplehydrology_amd/csrc/shy_device.hpp): for each size given as
// "nx ny" pairs, with and without blocks, every cell has its own index below
// tile_cells, tile_xy maps it back, unused indices map outside the map and are
// at most 1/16 of the cells, and (with full 64 x 64 blocks) a tile of 4096
// indices is a 64 x 64 square whose 32-index lines are 4 x 8 cells.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../simplehydrology_amd/csrc/shy_device.hpp"

int main(int argc, char** argv) {
  long long checked = 0, bad = 0;
  for (int a = 1; a + 1 < argc; a += 2)
    for (int blocks = 0; blocks < 2; ++blocks) {
      const int nx = std::atoi(argv[a]), ny = std::atoi(argv[a + 1]);
      const shy::TileMap m = shy::tile_map(nx, ny, blocks != 0);
      const long long n = shy::tile_cells(m, nx, ny);
      if (n < (long long)nx * ny || 16 * n > 17LL * nx * ny) ++bad;
      std::vector<char> used(n, 0);
      for (int x = 0; x < nx; ++x)
        for (int y = 0; y < ny; ++y) {
          const int i = shy::tile_index(m, x, y);
          ++checked;
          if (i < 0 || i >= n || used[i]) { ++bad; continue; }
          used[i] = 1;
          int u, v;
          shy::tile_xy(m, i, u, v);
          if (u != x || v != y) ++bad;
          if (m.a == 6 && m.b == 6) {
            const int c = shy::tile_index(m, x & ~63, y & ~63), l = shy::tile_index(m, x & ~3, y & ~7);
            if (i >> 12 != c >> 12 || i >> 5 != l >> 5 || (l & 31) || (c & 4095)) ++bad;
          }
          if (!blocks && i != x * ny + y) ++bad;
        }
      for (long long i = 0; i < n; ++i) {
        int u, v;
        shy::tile_xy(m, (int)i, u, v);
        if (!used[i] && u < nx && v < ny) ++bad;
      }
    }
  std::printf("cells %lld mismatches %lld\n", checked, bad);
  return bad ? 1 : 0;
}
