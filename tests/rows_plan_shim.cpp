// Test shim: the row kernel's host-side rules (gartus_amd/csrc/rows_plan.h) through a C ABI.
// Built by tests/test_rows_plan.py with g++.
#include "../gartus_amd/csrc/rows_plan.h"

extern "C" int shim_rows_frags(int ca, int cb, int cout, int grad, int64_t tiles) {
  return gdn::rows_frags(ca, cb, cout, grad != 0, tiles);
}
