// watch_wait.hpp -- the host's wait on a watched run's two words: [0] steps
// begun, [1] 1 once a step was the identity.  No HIP: the stream is a query.
#pragma once

#include <cstdint>

namespace abm {

enum class StreamState { kRunning, kIdle, kFailed };
enum class Waited { kBegun, kSettled, kFailed, kSilent };

// Waits until step `begun` (counted from 1) has begun, or one was the identity.
// query() is asked now and then: a stream that failed ends the wait, and so does
// an idle one.  An identity step may tell [1] alone, and the host may be held up
// between its reads and the query for as long as the steps launched ahead take:
// so both words are read again once the stream is idle, when every store has
// arrived, and only then is a run that told neither kSilent.
template <class Query>
inline Waited wait_watch(const int32_t *watch, int32_t begun, Query query) {
  for (uint32_t spin = 0;; ++spin) {
    if (__atomic_load_n(&watch[1], __ATOMIC_RELAXED)) return Waited::kSettled;
    if (__atomic_load_n(&watch[0], __ATOMIC_RELAXED) >= begun) return Waited::kBegun;
    if ((spin & 0x3FFF) != 0x3FFF) continue;
    const StreamState state = query();
    if (state == StreamState::kRunning) continue;
    if (state == StreamState::kFailed) return Waited::kFailed;
    if (__atomic_load_n(&watch[1], __ATOMIC_ACQUIRE)) return Waited::kSettled;
    return __atomic_load_n(&watch[0], __ATOMIC_ACQUIRE) >= begun ? Waited::kBegun
                                                                  : Waited::kSilent;
  }
}

}  // namespace abm
