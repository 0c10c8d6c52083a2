// ccd_dispatch.cpp -- selects the compiled CCD kernel shape at run time
// (the shapes are listed in ccd_shapes.h, each built in its own unit).
#include <hip/hip_runtime.h>

#include "ccd_core.h"
#include "ccd_kernel.h"
#include "ccd_shapes.h"

namespace c2a {

bool kernel_shape_ok(int K, int CAP, int NW, int V) {
#define C2A_OK_CASE(k, cap, nw, v) \
  if (K == k && CAP == cap && NW == nw && V == v) return true;
  C2A_SHAPES(C2A_OK_CASE)
#undef C2A_OK_CASE
  return false;
}

int kernel_blocks_per_cu(int K, int CAP, int NW, int V) {
#define C2A_OCC_CASE(k, cap, nw, v) \
  if (K == k && CAP == cap && NW == nw && V == v) \
    return occupancy_shape<k, cap, nw, v>();
  C2A_SHAPES(C2A_OCC_CASE)
#undef C2A_OCC_CASE
  return 0;
}

hipError_t launch_ccd(const KArgs& a, int K, int CAP, int NW, int blocks, hipStream_t s) {
  const bool fixed = a.mode == MODE_CONTACT || a.mode == MODE_DISTANCE;
  const int V = a.scorer.on != 0 ? 1 : (fixed && kernel_shape_ok(K, CAP, NW, 2) ? 2 : 0);
#define C2A_LAUNCH_CASE(k, cap, nw, v)                       \
  if (K == k && CAP == cap && NW == nw && V == v) \
    return launch_shape<k, cap, nw, v>(a, blocks, s);
  C2A_SHAPES(C2A_LAUNCH_CASE)
#undef C2A_LAUNCH_CASE
  return hipErrorInvalidValue;
}

}  // namespace c2a
