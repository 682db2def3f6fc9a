// Choice of a batch's launch shape from measured times (host code, no HIP
// types: batched.hip and the CPU checks share it).
#pragma once

namespace ccpi {

// Launch shape of a batch: slices per BP item (rc) and the grids of the FP
// items outside the shared walk and of the BP: 0 launches one wavefront per
// FP item and one workgroup per BP item (the dispatcher balances the uneven
// items), a positive value is a persistent grid of that many workgroups
// (capped at residency) that deals the items out by a fixed stride.
struct Tuned {
  int rc;
  int fp_grid;
  int bp_grid;
};

// The fastest of 8 and 16 slices per BP item and of 0, 2, 4 and 8 workgroups
// per CU for each projector.  fp_ms(grid) and bp_ms(grid) time one launch;
// bp_items(rc) lays the items out for rc slices before bp_ms is asked.  The
// shared walk has neither rc nor a grid to choose, and the other FP items no
// rc: the BP's times alone decide on rc, and without such items (fp_items
// false) no FP is run.
template <class Items, class FpMs, class BpMs>
Tuned tune_batch(bool fp_items, int cus, Items &&bp_items, FpMs &&fp_ms, BpMs &&bp_ms) {
  Tuned best{16, 0, 0};
  float bp_best = 1e30f;
  for (int rc : {8, 16}) {
    bp_items(rc);
    for (int per_cu : {0, 2, 4, 8}) {
      const float ms = bp_ms(per_cu * cus);
      if (ms < bp_best) {
        bp_best = ms;
        best.rc = rc;
        best.bp_grid = per_cu * cus;
      }
    }
  }
  float fp_best = 1e30f;
  if (fp_items)
    for (int per_cu : {0, 2, 4, 8}) {
      const float ms = fp_ms(per_cu * cus);
      if (ms < fp_best) {
        fp_best = ms;
        best.fp_grid = per_cu * cus;
      }
    }
  return best;
}

}  // namespace ccpi
