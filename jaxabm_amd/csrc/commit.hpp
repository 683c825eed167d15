// commit.hpp -- the end of a replayed step, shared by the kernels that run it:
// result copies, then the step's counters and the next step's keys.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "jaxabm_amd.h"

namespace abm {

// A step's result copies: item y copies items.it[y].bytes from src to dst +
// row * row_stride (row read from device memory when row_stride != 0; rows at
// or past row_limit are not written).  The list travels by value in the kernel
// arguments, so a captured launch keeps it.
struct CopyItems {
  abm_copy_item it[ABM_MAX_COPY_ITEMS];
};

struct CommitTail {
  int64_t *row;
  int32_t *ts;
  uint32_t *done;
  const uint32_t *key_table;
  int64_t key_rows;
  int32_t key_words;
  uint32_t *key_dst;
};

// One item by threads first, first + step, ...
__device__ __forceinline__ void commit_copy(const abm_copy_item &c, const int64_t *row,
                                            int64_t first, int64_t step) {
  int64_t r = 0;
  if (c.row_stride != 0) {
    r = row[0];
    if (r < 0 || r >= c.row_limit) return;
  }
  char *dst = (char *)c.dst + r * c.row_stride;
  const char *src = (const char *)c.src;
  if ((((uintptr_t)dst | (uintptr_t)src | (uintptr_t)c.bytes) & 15u) == 0) {
    const int64_t n16 = c.bytes >> 4;
    for (int64_t i = first; i < n16; i += step) ((uint4 *)dst)[i] = ((const uint4 *)src)[i];
  } else {
    for (int64_t i = first; i < c.bytes; i += step) dst[i] = src[i];
  }
}

// What a thread of the first wavefront needs to end the step, loaded before the
// workgroup's own work so that nothing but stores follows the last arrival.
struct CommitNext {
  int64_t row;   // the new row
  int32_t ts;
  uint32_t key;  // word `lane` of the new row's keys
};

__device__ __forceinline__ CommitNext commit_begin(const CommitTail &t) {
  CommitNext n{0, 0, 0u};
  if (threadIdx.x >= 64) return n;
  n.row = t.row[0] + 1;
  n.ts = t.ts[0] + 1;
  if (t.key_dst && n.row < t.key_rows && (int32_t)threadIdx.x < t.key_words)
    n.key = t.key_table[n.row * t.key_words + threadIdx.x];
  return n;
}

// Called by every workgroup (all its threads) once it has read row; the last of
// `total` to arrive advances row and ts, returns `done` to 0, and copies row
// r + 1 of the key table to key_dst for the next step (if r + 1 < key_rows).
// The counter orders reads of row before its write and nothing else: what the
// workgroups wrote becomes visible with the kernel's end, so no fence (which
// would write the caches back, 1 us and more) is needed.
__device__ __forceinline__ void commit_arrive(const CommitTail &t, const CommitNext &n,
                                              uint32_t total) {
  __syncthreads();  // every thread's read of row has returned
  if (threadIdx.x >= 64) return;
  uint32_t before = 0;
  if (threadIdx.x == 0)
    before =
        __hip_atomic_fetch_add(t.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__shfl(before, 0) != total - 1) return;
  if (threadIdx.x == 0) {
    t.row[0] = n.row;
    t.ts[0] = n.ts;
    *t.done = 0u;
  }
  if (t.key_dst && n.row < t.key_rows) {
    if ((int32_t)threadIdx.x < t.key_words) t.key_dst[threadIdx.x] = n.key;
    for (int32_t w = 64 + (int32_t)threadIdx.x; w < t.key_words; w += 64)
      t.key_dst[w] = t.key_table[n.row * t.key_words + w];
  }
}

inline int check_commit(const abm_copy_item *items, int32_t n_items, const CommitTail &t,
                        CopyItems *list, int64_t *max_bytes, const char *who) {
  if (!((items || n_items == 0) && n_items >= 0 && n_items <= ABM_MAX_COPY_ITEMS && t.row &&
        t.ts && t.done && t.key_rows >= 0 && t.key_words >= 0 &&
        (!t.key_dst || (t.key_table && t.key_words > 0)))) {
    set_error(std::string(who) + ": bad arguments");
    return kErrInvalid;
  }
  *max_bytes = 0;
  for (int32_t i = 0; i < n_items; ++i) {
    const abm_copy_item &c = items[i];
    if (!(c.src && c.dst && c.bytes >= 0 && (c.row_stride == 0 || c.row_limit > 0))) {
      set_error(std::string(who) + ": bad item");
      return kErrInvalid;
    }
    list->it[i] = c;
    if (c.bytes > *max_bytes) *max_bytes = c.bytes;
  }
  return kOk;
}

}  // namespace abm
