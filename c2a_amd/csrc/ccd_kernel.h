// ccd_kernel.h -- launcher of the gfx950 CCD kernel.
#pragma once

#include <hip/hip_runtime.h>

#include "ccd_types.h"

namespace c2a {

// The shapes of ccd_shapes.h: K = speculative subtree depth, CAP = DFS stack
// capacity in entries, NW = wavefronts per query, V = variant.  launch_ccd takes
// the learned order's variant when a.scorer.on, and the contact and distance
// variant for those modes where it exists.
bool kernel_shape_ok(int K, int CAP, int NW, int V);
hipError_t launch_ccd(const KArgs& a, int K, int CAP, int NW, int blocks, hipStream_t s);
int kernel_blocks_per_cu(int K, int CAP, int NW, int V);

}  // namespace c2a
