// How a launch's workgroups are laid over a grid (host arithmetic, no HIP
// types: the launchers and the CPU checks share it).
#pragma once

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

}  // namespace ccpi
