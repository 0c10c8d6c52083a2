// static_kernel.h -- launcher of the static-query kernel (static_kernel.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "static_query.h"

namespace c2a {

// Threads per workgroup; the workspace holds blocks * kStaticBlock slices.
constexpr int kStaticBlock = 256;

hipError_t launch_static(const StaticArgs& a, int blocks, hipStream_t s);

// One wavefront per query (static_wave.h): whether it takes the query, the
// workspace of one wavefront, and the launch (blocks wavefronts).
bool static_wave_ok(int kind, int qsize, int pair_cap, int depth_sum);
int64_t static_wave_bytes(int kind, int pair_cap, int depth_sum);
hipError_t launch_static_wave(const StaticArgs& a, int blocks, hipStream_t s);

}  // namespace c2a
