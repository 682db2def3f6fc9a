// CPU checks of the library's host rules (csrc headers without HIP types).
// host_rules <check> exits 0 where the check holds; test_host_rules.py builds
// and runs it.
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "grid.hpp"

static int failed = 0;
#define EXPECT(c) \
  do { \
    if (!(c)) { \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); \
      failed = 1; \
    } \
  } while (0)

// No dimension of a grid reaches 2^32 threads, every workgroup has a number,
// the numbers stay below 2^31, and a row starts on the first XCD.
static void grids() {
  const long long top = (1LL << 31) - (1LL << ccpi::kGridRowBits);
  for (int threads : {64, 128, 192, 256, 320, 576, 1024}) {
    const long long edge = (1LL << 32) / threads;
    for (long long blocks : {1LL, 8LL, 4096LL, edge - 1, edge, edge + 1, 3 * edge, top - 1}) {
      if (blocks >= top) continue;
      const ccpi::WgGrid G = ccpi::wg_grid(blocks, threads);
      EXPECT(G.x > 0 && G.y > 0);
      EXPECT((long long)G.x * threads < (1LL << 32) && G.y < 65536);
      EXPECT((long long)G.x * G.y >= blocks && (long long)G.x * G.y < (1LL << 31));
      EXPECT(G.y == 1 || (G.x == 1u << ccpi::kGridRowBits && G.x % ccpi::kXcds == 0));
      EXPECT(G.y > 1 || G.x == blocks);
    }
    EXPECT(ccpi::wg_grid(top, threads).x == 0);
  }
}

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "grids")) grids();
  else return 2;
  return failed;
}
