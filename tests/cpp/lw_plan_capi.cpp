// The LWEnKF update's workspace plan behind a C function.
#include "mda_internal.hpp"

extern "C" int64_t lw_plan_ntap(int k, int64_t n, int64_t p) {
  return mda::lw_update_plan(k, n, p).ntap;
}
