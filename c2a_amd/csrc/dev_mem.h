// dev_mem.h -- the library's device allocations.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace c2a {

// hipMalloc that gives up the memory the library keeps between calls before it
// fails (capi.cpp).
hipError_t device_malloc(void** p, size_t n);

}  // namespace c2a
