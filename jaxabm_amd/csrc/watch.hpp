// watch.hpp -- runs whose kernels tell the host how far they are: two words of
// pinned host memory, [0] steps begun, [1] 1 once a step was the identity.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "common.hpp"
#include "jaxabm_amd.h"

namespace abm {

__device__ __forceinline__ void tell_host(int32_t *p, int32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

inline void clear_watch(int32_t *watch) {
  __atomic_store_n(&watch[0], 0, __ATOMIC_RELAXED);
  __atomic_store_n(&watch[1], 0, __ATOMIC_RELEASE);
}

// Waits until step `begun` (counted from 1) has begun, or one was the identity.
// An error of the stream ends the wait, and so does a stream that has finished
// without saying so.
inline int wait_begun(const int32_t *watch, int32_t begun, hipStream_t s, const char *who,
                      bool *settled) {
  for (uint32_t spin = 0;; ++spin) {
    *settled = __atomic_load_n(&watch[1], __ATOMIC_RELAXED) != 0;
    if (*settled || __atomic_load_n(&watch[0], __ATOMIC_RELAXED) >= begun) return kOk;
    if ((spin & 0x3FFF) != 0x3FFF) continue;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    if (e != hipSuccess) return hip_fail(e, who);
    if (__atomic_load_n(&watch[0], __ATOMIC_ACQUIRE) >= begun) return kOk;
    set_error(std::string(who) + ": watch must be host memory the device can write");
    return kErrInvalid;
  }
}

}  // namespace abm
