// How a launch's workgroups are laid over a grid and over a CU's LDS (host
// arithmetic, no HIP types: the launchers and the CPU checks share it).
#pragma once

#include <algorithm>
#include <cstddef>

namespace ccpi {

constexpr int kXcds = 8;

// Workgroups 0 .. blocks - 1 of `threads` threads as a grid of x by y.  HIP
// takes fewer than 2^32 threads along one dimension, so a launch of more goes
// over both; its workgroups are numbered blockIdx.x + (blockIdx.y <<
// kGridRowBits) (wg_index), which is the order they are dispatched in, and a
// row is a multiple of the XCDs, so number modulo 8 stays the XCD.  The last
// row is whole: numbers from `blocks` on are the kernel's to leave out.  x = 0:
// too many workgroups for their numbers to fit an int.
constexpr int kGridRowBits = 20;
struct WgGrid {
  unsigned x, y;
};
inline WgGrid wg_grid(long long blocks, int threads) {
  constexpr long long row = 1LL << kGridRowBits;
  static_assert(row % kXcds == 0, "a row starts on the first XCD");
  if (blocks >= (1LL << 31) - row) return {0, 0};
  if (blocks * threads < (1LL << 32)) return {(unsigned)blocks, 1};
  return {(unsigned)row, (unsigned)((blocks + row - 1) / row)};
}

// Ray tiles of the cone FP: consecutive workgroups of one XCD take a tile of
// adjacent angles x adjacent rays, whose walks cross mostly the same columns
// at the same time, so the columns are read from that XCD's L2.  512^3, ms
// per FP and bytes fetched from beyond L2: rays dealt to the XCDs in turn
// 83 / 601 GB; tiles of 16 x 16 67.7, 1 x 64 78.4, 8 x 32 72.7, 32 x 8 66.1;
// with the loads as they are now 32 x 8 60.8, 64 x 8 60.0 / 203 GB, 128 x 8
// 59.7, 128 x 4 60.6; 256^3 4.07 to 4.10 for all four.
// A tile has at most kFpTileA angles, and fewer where that leaves an XCD less
// than kFpTiles tiles: with 64 angles, 58 angles x 13 columns were one tile
// each for four XCDs and none for the others (64 x 130 x 12, 447 rows 0.0189
// ms before the tiles, 0.0253 with 64 angles, 0.0156 now), 103 x 19 columns 3
// for some and 2 for others (57 x 62 x 29, 515 rows 0.025, 0.028, 0.020).
constexpr int kFpTileA = 64, kFpTileH = 8, kFpTiles = 16;
struct RayTiles {
  int angles;        // per tile
  long long tiles;
};
inline RayTiles cone_fp_tiles(int na, int nh) {
  const int nth = (nh - 1) / kFpTileH + 1;
  const int nta = std::max((na - 1) / kFpTileA + 1,
                           std::min(na, (kXcds * kFpTiles - 1) / nth + 1));
  const int angles = (na - 1) / nta + 1;
  return {angles, (long long)((na - 1) / angles + 1) * nth};
}

// The column block of place p in the parallel FP's row `ta` of tiles, nb column
// blocks a row.  Tiles go to the XCDs in turn, so with p itself and nb a
// multiple of 8 a block stays on one XCD, with 4 blocks on two, and where the
// volume's shadow takes the middle of the detector the XCDs of the outer blocks
// run dry.  Such rows are turned, each by 3 places more than the one before or,
// of 4 blocks, by one: 80 x 80 x 30, 300 angles, 500 columns 0.084 ms unturned,
// 0.050 by one and by three; 200 x 200 x 52, 42 angles, 500 columns 0.102, 0.097,
// 0.073; 250 x 250 x 30, 180 angles, 512 columns 0.167, 0.130, 0.116; 420 x 420 x
// 20, 300 angles, 500 columns 0.386, 0.347, 0.360; 84 x 20 x 21, 145 angles, 244
// columns 0.049, 0.038.  Others meet every XCD, or, 12 blocks, enough of them:
// 512 x 512 x 32, 360 angles, 725 columns 0.678, turned by one 0.681, by seven
// 0.70; 147 x 147 x 61, 72 angles, 588 columns 0.067, turned 0.070 to 0.087.
constexpr int par_tile_column(int nb, int ta, int p) {
  if (nb != 4 && nb % 8 != 0) return p;
  const int c = p + (ta % nb) * (nb == 4 ? 1 : 3) % nb;
  return c < nb ? c : c - nb;
}

// LDS of the parallel tiled BP per angle of a block, two blocks: hmax columns
// of `slices` rows, their positions and the span.
inline std::size_t par_bp_angle_bytes(int hmax, int slices) {
  return 2 * ((std::size_t)hmax * (sizeof(float) * slices + sizeof(double)) + 2 * sizeof(int));
}
// LDS of one workgroup: the blocks and the spans of 256 angles.
inline std::size_t par_bp_tile_bytes(int hmax, int slices, int ab) {
  return par_bp_angle_bytes(hmax, slices) * (std::size_t)ab + 256 * 2 * sizeof(int);
}
// Angles per block: at most 4 (a wavefront stages one each), and as many as
// leave the CU's 160 KB, handed out in units of 1280 bytes, for the five
// workgroups that the registers allow (128 bytes are the norm's); or else one.
// With 32 KB of blocks only four fitted where pixels are half a voxel or a
// quarter with 8 slices: 237 x 237 x 13, 133 angles, pixels of half a voxel
// 0.106 ms before there were two blocks, 0.121 with four angles (30016 bytes),
// 0.099 with three; 458 x 224 x 2, 317 angles, a quarter 0.44, 0.53, 0.42.
// Fewer than fit lose: 566 x 566 x 16, 73 angles, a quarter 0.52 with two (27968
// bytes), 0.56 with one.
constexpr std::size_t kParBpLds = 25 * 1280;
inline int par_bp_block_angles(int hmax, int slices) {
  int n = 4;
  while (n > 1 && par_bp_tile_bytes(hmax, slices, n) + 128 > kParBpLds) n--;
  return n;
}

}  // namespace ccpi
