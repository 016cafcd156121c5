// Test shim: the row kernel's host-side rules (gartus_amd/csrc/rows_plan.h) through a C ABI.
// Built by tests/test_rows_plan.py with g++.
#include "../gartus_amd/csrc/rows_plan.h"

extern "C" int shim_rows_frags(int ca, int cb, int cout, int grad, int64_t tiles) {
  return gdn::rows_frags(ca, cb, cout, grad != 0, tiles);
}

extern "C" void shim_rows_split(int n, int h, int w, int groups, int waves, int out[4]) {
  const gdn::RowsSplit s = gdn::rows_split(n, h, w, groups, waves);
  out[0] = s.rows;
  out[1] = s.segs;
  out[2] = s.strips;
  out[3] = s.blocks;
}
