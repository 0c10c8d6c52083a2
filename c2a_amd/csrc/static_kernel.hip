// static_kernel.hip -- the static proximity queries on gfx950: one wavefront
// per query where static_wave.h takes the search, else one thread per query
// (static_query.h).  Both take queries from a device work queue until it
// drains, each wavefront or thread with its own slice of the workspace.
#include <hip/hip_runtime.h>

#include "static_query.h"
#include "static_wave.h"
#include "static_kernel.h"

namespace c2a {

__global__ void static_zero_counter(int64_t* c) { *c = 0; }

__global__ void __launch_bounds__(kStaticBlock) static_kernel(StaticArgs a) {
  const int64_t tid = (int64_t)blockIdx.x * kStaticBlock + threadIdx.x;
  SqEntry* ws = a.ws + tid * a.ws_entries;
  for (;;) {
    const int64_t qi =
        (int64_t)atomicAdd(reinterpret_cast<unsigned long long*>(a.counter), 1ull);
    if (qi >= a.nq) break;
    static_query(a, qi, ws);
  }
}

// One wavefront per query, taken from the same work queue.
template <int KIND>
__global__ void __launch_bounds__(64) static_wave_kernel(StaticArgs a) {
  __shared__ SqWaveLds g;
  const int lane = threadIdx.x;
  unsigned char* ws = a.wave_ws + (int64_t)blockIdx.x * a.wave_bytes;
  for (;;) {
    if (lane == 0)
      g.ticket = (int64_t)atomicAdd(reinterpret_cast<unsigned long long*>(a.counter), 1ull);
    lane_sync();
    const int64_t qi = lane0_bcast64(g.ticket);
    lane_sync();
    if (qi >= a.nq) break;
    sq_wave_query<KIND>(a, qi, g, ws, lane);
  }
}

bool static_wave_ok(int kind, int qsize, int pair_cap, int depth_sum) {
  return depth_sum <= kSqWaveDepth &&
         ((kind == SQ_COLLIDE && pair_cap <= kSqWavePairs) ||
          (kind == SQ_TOLERANCE && qsize <= 2) || kind == SQ_DISTANCE_CS);
}
int64_t static_wave_bytes(int kind, int pair_cap, int depth_sum) {
  return sq_wave_bytes(kind, depth_sum, pair_cap);
}

hipError_t launch_static_wave(const StaticArgs& a, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(static_zero_counter, dim3(1), dim3(1), 0, s, a.counter);
  auto fn = a.kind == SQ_COLLIDE     ? static_wave_kernel<SQ_COLLIDE>
            : a.kind == SQ_TOLERANCE ? static_wave_kernel<SQ_TOLERANCE>
                                     : static_wave_kernel<SQ_DISTANCE_CS>;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_static(const StaticArgs& a, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(static_zero_counter, dim3(1), dim3(1), 0, s, a.counter);
  hipLaunchKernelGGL(static_kernel, dim3(blocks), dim3(kStaticBlock), 0, s, a);
  return hipGetLastError();
}

}  // namespace c2a
