// CPU checks of the library's host rules (csrc headers without HIP types).
// host_rules <check> exits 0 where the check holds; test_host_rules.py builds
// and runs it.
#include <atomic>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <memory>
#include <thread>
#include <vector>

#include "batch_tune.hpp"
#include "grid.hpp"
#include "kept.hpp"

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

// Live rays of the cone FP per XCD: where there are enough rays to share, no
// XCD has much more than its share of the rays with the last column tile full.
static void cone_tiles() {
  for (int na : {1, 5, 33, 58, 64, 65, 90, 103, 146, 194, 360, 720})
    for (int nh : {2, 9, 13, 17, 19, 64, 96, 283, 384, 768}) {
      const ccpi::RayTiles T = ccpi::cone_fp_tiles(na, nh);
      const int nth = (nh + ccpi::kFpTileH - 1) / ccpi::kFpTileH;
      EXPECT(T.angles >= 1 && T.angles <= ccpi::kFpTileA && T.tiles % nth == 0);
      EXPECT(T.tiles / nth * T.angles >= na && (T.tiles / nth - 1) * T.angles < na);
      long long per[ccpi::kXcds] = {}, most = 0;
      for (long long t = 0; t < T.tiles; t++) {
        const long long a0 = t / nth * T.angles, h0 = t % nth * ccpi::kFpTileH;
        per[t % ccpi::kXcds] += std::min<long long>(T.angles, na - a0) *
                                std::min<long long>(ccpi::kFpTileH, nh - h0);
      }
      for (long long p : per) most = std::max(most, p);
      if ((long long)na * nth >= ccpi::kXcds * ccpi::kFpTiles)
        EXPECT(most * ccpi::kXcds <= 1.15 * na * nth * ccpi::kFpTileH);
    }
}

// Every row of the parallel FP's tiles holds every column block once, and where
// a block would keep to one or two XCDs and the middle half of the blocks
// holds the work, no XCD has more than 1.5 times its share of it in 24 rows.
static void par_columns() {
  for (int nb = 1; nb <= 70; nb++) {
    long long per[ccpi::kXcds] = {}, all = 0;
    for (int ta = 0; ta < 24; ta++) {
      std::vector<int> seen(nb);
      for (int p = 0; p < nb; p++) {
        const int c = ccpi::par_tile_column(nb, ta, p);
        EXPECT(c >= 0 && c < nb);
        if (c < 0 || c >= nb) return;
        seen[c]++;
        const bool middle = 4 * c >= nb - 1 && 4 * c <= 3 * nb - 1;
        per[((long long)ta * nb + p) % ccpi::kXcds] += middle;
        all += middle;
      }
      for (int s : seen) EXPECT(s == 1);
    }
    if (nb % 4 == 0)
      for (long long p : per) EXPECT(2 * p * ccpi::kXcds <= 3 * all);
  }
  EXPECT(ccpi::par_tile_column(1 << 25, (1 << 26) + 3, (1 << 25) - 1) < 1 << 25);
  EXPECT(ccpi::par_tile_column(1 << 25, (1 << 26) - 1, 0) >= 0);
}

// The tiled parallel BP's blocks leave room for five workgroups on a CU (160 KB,
// handed out 1280 bytes at a time, with 128 bytes of the kernel's own) wherever
// more than one angle is staged, and no angle less than fits is staged.
static void bp_blocks() {
  for (int slices : {8, 16})
    for (int hmax = 7; hmax <= 1023; hmax++) {
      const int ab = ccpi::par_bp_block_angles(hmax, slices);
      auto five = [&](int n) {
        return 5 * ((ccpi::par_bp_tile_bytes(hmax, slices, n) + 128 + 1279) / 1280 * 1280) <=
               160 * 1024;
      };
      EXPECT(ab >= 1 && ab <= 4);
      EXPECT(ab == 1 || five(ab));
      EXPECT(ab == 4 || !five(ab + 1));
    }
}

struct Thing {
  static std::atomic<int> live;
  int id;
  size_t size;
  std::atomic<int> holders{0};
  Thing(int i, size_t s) : id(i), size(s) { live++; }
  ~Thing() { live--; }
  size_t bytes() const { return size; }
};
std::atomic<int> Thing::live{0};
using Things = ccpi::Kept<Thing>;
static std::unique_ptr<Thing> thing(int id, size_t size) {
  return std::make_unique<Thing>(id, size);
}

// At most 4 and 100 bytes stay, the ones left last; each device its own.
static void kept() {
  Things k(4, 100);
  EXPECT(!k.take(0));
  for (int i = 0; i < 7; i++) {
    k.leave(0, thing(i, 10));
    EXPECT(Thing::live == (i < 4 ? i + 1 : 4));
  }
  EXPECT(!k.take(1));
  for (int i = 6; i >= 3; i--) {
    auto t = k.take(0);
    EXPECT(t && t->id == i);
  }
  EXPECT(!k.take(0) && Thing::live == 0);
  // over the bytes together: the older ones go, a small older one may stay
  k.leave(0, thing(0, 20));
  k.leave(0, thing(1, 60));
  k.leave(1, thing(2, 50));
  EXPECT(Thing::live == 2);
  auto a = k.take(0);
  EXPECT(a && a->id == 0);
  auto b = k.take(1);
  EXPECT(b && b->id == 2);
  // one larger than the limit never stays, one of the limit does, alone
  k.leave(0, std::move(a));
  k.leave(0, thing(3, 101));
  EXPECT(Thing::live == 2);
  k.leave(0, thing(4, 100));
  EXPECT(Thing::live == 2);   // 4 and the held b
  k.leave(1, std::move(b));
  EXPECT(Thing::live == 1);
  k.give_back();
  EXPECT(Thing::live == 0 && !k.take(0) && !k.take(1));
}

// No object has two holders, and no more than the limit stay.
static void kept_threads() {
  Things k(4, 1000);
  std::atomic<bool> shared{false};
  std::vector<std::thread> ts;
  for (int n = 0; n < 8; n++)
    ts.emplace_back([&, n] {
      for (int i = 0; i < 2000; i++) {
        auto t = k.take(i % 2);
        if (!t) t = thing(n, 10 + n);
        if (t->holders++ != 0) shared = true;
        std::this_thread::yield();
        t->holders--;
        k.leave(i % 2, std::move(t));
        if (i % 500 == 499) k.give_back();
      }
    });
  for (auto &t : ts) t.join();
  EXPECT(!shared && Thing::live <= 4);
  k.give_back();
  EXPECT(Thing::live == 0);
}

// A refused allocation is tried once more, after what idles has gone back;
// another error is not.
static void refused_allocation() {
  enum Status { kOk, kRefused, kOther };
  Things k(4, 1000);
  auto fill = [&] {
    for (int i = 0; i < 3; i++) k.leave(0, thing(i, 10));
  };
  int tries = 0;
  auto back = [&] { k.give_back(); };
  auto room = [&] {
    tries++;
    return Thing::live == 0 ? kOk : kRefused;
  };
  fill();
  EXPECT(ccpi::alloc_giving_back(kRefused, room, back) == kOk && tries == 2);
  EXPECT(ccpi::alloc_giving_back(kRefused, room, back) == kOk && tries == 3);
  fill();
  auto held = k.take(0);
  EXPECT(ccpi::alloc_giving_back(kRefused, room, back) == kRefused && tries == 5);
  EXPECT(Thing::live == 1);   // the held one is not touched
  fill();
  EXPECT(ccpi::alloc_giving_back(kRefused, [] { return kOther; }, back) == kOther);
  EXPECT(Thing::live == 4);
}

// The BP's times alone choose the slices per item, whatever the FP's are; the
// FP's grid is timed once each, and only where there are items to time.
static void batch_tune() {
  int rc = 0, fp_runs = 0;
  // 16 slices are faster, at 4 workgroups per CU
  auto bp = [&](int grid) { return (rc == 16 ? 7.0f : 8.0f) + (grid == 4 * 256 ? 0.f : 0.5f); };
  auto items = [&](int r) { rc = r; };
  for (bool have : {false, true})
    for (float noise : {0.f, 100.f}) {
      fp_runs = 0;
      // an FP that was timed beside 16 slices would have spoilt them
      auto fp = [&](int grid) {
        fp_runs++;
        return 9.0f + (rc == 16 ? noise : 0.f) + (grid == 2 * 256 ? 0.f : 1.f);
      };
      const ccpi::Tuned T = ccpi::tune_batch(have, 256, items, fp, bp);
      EXPECT(T.rc == 16 && T.bp_grid == 4 * 256);
      EXPECT(fp_runs == (have ? 4 : 0));
      EXPECT(T.fp_grid == (have ? 2 * 256 : 0));
    }
  // no persistent grid where one workgroup per item is as fast
  const ccpi::Tuned T =
      ccpi::tune_batch(true, 256, items, [](int) { return 1.f; }, [](int) { return 1.f; });
  EXPECT(T.rc == 8 && T.fp_grid == 0 && T.bp_grid == 0);
}

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "grids")) grids();
  else if (!std::strcmp(what, "cone_tiles")) cone_tiles();
  else if (!std::strcmp(what, "par_columns")) par_columns();
  else if (!std::strcmp(what, "bp_blocks")) bp_blocks();
  else if (!std::strcmp(what, "kept")) kept();
  else if (!std::strcmp(what, "kept_threads")) kept_threads();
  else if (!std::strcmp(what, "refused_allocation")) refused_allocation();
  else if (!std::strcmp(what, "batch_tune")) batch_tune();
  else return 2;
  return failed;
}
