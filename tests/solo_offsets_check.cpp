// Host check of the record offsets of the walk of one wave per drop (solo_rec,
// solo_off, solo_terrain in simplehydrology_amd/csrc/shy_device.hpp): for each
// terrain size given as "nx ny" pairs that solo_terrain takes, the 32-bit offset of
// every cell (of large maps the first and last 4 rows, and columns of the rest)
// is 32 bytes times pack_rec in 64 bits, and the factors fit the 24-bit product.
// Prints per size whether it is taken; exits 1 on any mismatch.
#include <cstdio>
#include <cstdlib>

#include "../simplehydrology_amd/csrc/shy_device.hpp"

int main(int argc, char** argv) {
  long long bad = 0;
  for (int a = 1; a + 1 < argc; a += 2) {
    const int nx = std::atoi(argv[a]), ny = std::atoi(argv[a + 1]);
    const bool take = shy::solo_terrain(nx, ny);
    std::printf("%d", take ? 1 : 0);
    if (!take) continue;
    const int s4 = shy::solo_stride4(ny);
    if (s4 >= 1 << 23 || (nx + 2) >> 1 >= 1 << 23) ++bad;
    const bool all = (long long)nx * ny < 4000000;
    for (int x = 0; x < nx; ++x)
      for (int y = 0; y < ny; ++y) {
        if (!all && x >= 4 && x < nx - 4 && y >= 2 && y < ny - 2) y = ny - 2;
        const uint64_t rec = ((uint64_t)(x >> 1) * (uint64_t)((ny + 1) >> 1) + (y >> 1)) * 4 +
                             (x & 1) * 2 + (y & 1);
        if ((uint64_t)shy::solo_off(shy::solo_rec(x, y, s4)) != 32 * rec) ++bad;
      }
  }
  std::printf("\n");
  return bad ? 1 : 0;
}
