// watch.hpp -- runs whose kernels tell the host how far they are: two words of
// pinned host memory, [0] steps begun, [1] 1 once a step was the identity.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "common.hpp"
#include "jaxabm_amd.h"
#include "watch_wait.hpp"

namespace abm {

__device__ __forceinline__ void tell_host(int32_t *p, int32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

inline void clear_watch(int32_t *watch) {
  __atomic_store_n(&watch[0], 0, __ATOMIC_RELAXED);
  __atomic_store_n(&watch[1], 0, __ATOMIC_RELEASE);
}

// wait_watch on a stream; *settled: one step was the identity.
inline int wait_begun(const int32_t *watch, int32_t begun, hipStream_t s, const char *who,
                      bool *settled) {
  hipError_t e = hipSuccess;
  const Waited w = wait_watch(watch, begun, [&] {
    e = hipStreamQuery(s);
    return e == hipSuccess         ? StreamState::kIdle
           : e == hipErrorNotReady ? StreamState::kRunning
                                   : StreamState::kFailed;
  });
  *settled = w == Waited::kSettled;
  if (w == Waited::kFailed) return hip_fail(e, who);
  if (w == Waited::kSilent) {
    set_error(std::string(who) + ": watch must be host memory the device can write");
    return kErrInvalid;
  }
  return kOk;
}

}  // namespace abm
