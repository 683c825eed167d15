// sir.hip -- network SIR step: synchronous S->I->R over an undirected CSR.
//
// Program semantics (reference schedule jaxabm/model.py:146-216, Network
// jaxabm/agentpy.py:530-615 rebuilt as CSR):
//   k_inf, k_rec = split(update_key)
//   u = uniform(k_inf, (nnz,)), r = uniform(k_rec, (n,))
//   S -> I  iff some CSR entry e of row v has old[col[e]] == I and u[e] < beta
//   I -> R  iff r[v] < gamma
// Counter-based draws let the kernel evaluate u[e] only for S-I entries and
// stop at the first infecting entry: the result is the same "any" as the dense
// formulation.  `u < p` is tested on the integer mantissa (m < ceil(p*2^23)),
// which is exact for the [0,1) uniform.
//
// Design for MI355X:
//  * Neighbour status comes from an infected-set bitmap (1 bit per agent,
//    125 KB at n = 1M, word count a multiple of 4) written by the previous
//    step.  Each of the 256 persistent 1024-thread blocks stages the whole
//    bitmap in LDS (160 KB per CU), so the random neighbour checks are LDS bit
//    tests instead of global gathers; graphs whose bitmap exceeds the LDS
//    budget read it from global memory (L2-resident) with the same kernel.
//    Staging costs a 125 KB read per block, so a block stages only when its
//    tile has many rows to scan (the epidemic peak) and otherwise tests bits
//    in the L2-resident global bitmap.
//  * A step whose previous step left no infected agent is the identity: the
//    kernel then only clears its bitmap spans and copies the counts.
//  * Work skipping with plain stores (no atomics): an agent u that is infected
//    after step s writes mark[w] = s + H (16-bit) into each neighbour w when
//    it was infected at s or (s + u) % H == 0.  At step t an S agent scans its
//    row only if (mark[v] - t) mod 2^16 <= H.  If v has a neighbour u infected
//    at the start of step t, u wrote a mark in some step s in [t-H, t-1] (its
//    infection step or its refresh phase) with value s + H in [t, t+H-1], and
//    later writes only store values in [t, t+H], so v is never skipped; stale
//    marks only cost a scan.  H = 16 with per-agent refresh phases cuts the
//    mark stores of long-lived infections by 16x without step-to-step spikes.
//  * Only its owner reads an agent's state byte, so state is updated in place
//    (an agent octet is written only when it changes); the bitmap is double-buffered (read
//    B[t&1], write B[(t+1)&1]) and each bitmap word is written whole by the
//    block owning its 64-agent span.
//  * The agent range is cut into 64-aligned chunks of equal (agents + degree
//    + heavy-row) cost and at most one tile, one per block.  A chunk is processed in tiles
//    of 8192 agents (eight per thread, loads issued together): S agents at risk go to an LDS
//    worklist; rows of degree <= 32 are scanned and marked by one lane (by
//    several in a tile of few rows), longer rows by wavefronts, 64 entries a unit.
//  * S/I/R counts: wave reductions -> LDS -> one atomic per block into one of
//    64 slots, reduced after the run.
//
// Layout (HBM): state uint8[n] (low 2 bits S=0/I=1/R=2, bit 2 = row degree
// > 32), mark uint16[n], bitmap uint32[2][words], row_ptr int32[n+1],
// col int32[nnz] (rows ascending), chunk_ptr int32[n_chunks+1].
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "common.hpp"
#include "jaxabm_amd.h"
#include "watch.hpp"

namespace abm {

constexpr int kSirThreads = 1024;
constexpr int kPerThread = 8;
constexpr int kTile = kSirThreads * kPerThread;
constexpr int kSirBlocks = 256;
constexpr int kHeavyDeg = 32;
constexpr int kChunkAlign = 64;
constexpr int64_t kChunkNodeCost = 4;
// extra chunk cost of a heavy row: a wavefront pays about two serial memory
// round trips per row whatever its degree
constexpr int64_t kChunkHeavyCost = 128;
constexpr int kChunksPerBlock = 1;
constexpr int kSlots = 64;                 // count slots per step
constexpr int kStepSlots = kSlots + 1;     // + one flag slot
constexpr int kStride = kStepSlots * 3;    // ints per step in the slots array
// slots[t][kSlots][1] = 1 when step t left an infected agent (plain stores
// of the same value by any block that has one): the next step reads this one
// word to decide whether it is the identity
constexpr int kLiveFlag = kSlots * 3 + 1;
constexpr uint8_t kHeavyBit = 4;
constexpr uint32_t kMarkHorizon = 16;
// a tile stages the bitmap in LDS when it has at least this many rows to scan
constexpr int32_t kStageItems = 512;
// LDS bitmap budget: 32768 words (1,048,576 agents, 128 KB)
constexpr int64_t kLdsBitmapWords = 32768;

struct SirStep {
  int64_t n, nnz;
  const int32_t *row_ptr, *col, *chunk_ptr;
  int32_t n_chunks;
  uint8_t *state;
  uint16_t *mark;
  const uint32_t *bm_in;
  uint32_t *bm_out;
  int64_t words;
  uint32_t t;
  const int32_t *prev_slots;  // previous step's count slots, or null
  const int32_t *prev2_slots; // the step before that, or null
  const uint32_t *keys;
  uint32_t thr_beta, thr_gamma;
  int32_t *slots;
  int32_t *watch;  // host memory, or null: [0] steps begun, [1] 1 once one was the identity
  int32_t begun;   // value for watch[0], or 0: this step does not tell
};

__device__ __forceinline__ bool infected(const uint32_t *__restrict__ bm, int32_t u) {
  return (bm[u >> 5] >> (u & 31)) & 1u;
}

__device__ __forceinline__ bool at_risk(uint16_t m, uint32_t t) {
  return (uint16_t)(m - (uint16_t)t) <= kMarkHorizon;
}

// Entries of a row that one lane loads per round, as two 16-byte loads: a
// lane's rows are scattered, so every load instruction of a wavefront touches
// 64 lines, and entry by entry the same lines were fetched again and again
// (they do not stay in the 32 KB L1).
constexpr int kRowRound = 8;

// c[k] = col[e + k] for e + k < hi, else -1.
__device__ __forceinline__ void load_row_round(const int32_t *__restrict__ col, int32_t e,
                                               int32_t hi, int64_t nnz, int32_t (&c)[kRowRound]) {
  if (e + kRowRound <= nnz) {
    int32_t v[kRowRound];
    __builtin_memcpy(v, col + e, 16);
    __builtin_memcpy(v + 4, col + e + 4, 16);
#pragma unroll
    for (int k = 0; k < kRowRound; ++k) c[k] = e + k < hi ? v[k] : -1;
  } else {  // the last entries of the array
#pragma unroll
    for (int k = 0; k < kRowRound; ++k) c[k] = e + k < hi ? col[e + k] : -1;
  }
}

// A row of degree <= 32 scanned by one lane: each round tests kRowRound
// entries and draws its S-I candidates in order, stopping at the first
// infecting one.
__device__ __forceinline__ bool scan_light(const int32_t *__restrict__ col,
                                           const uint32_t *__restrict__ bm, int32_t e, int32_t hi,
                                           Key kinf, int64_t nnz, uint32_t thr, int mode) {
  for (; e < hi; e += kRowRound) {
    int32_t c[kRowRound];
    load_row_round(col, e, hi, nnz, c);
    uint32_t cm = 0;
#pragma unroll
    for (int k = 0; k < kRowRound; ++k)
      if (c[k] >= 0 && infected(bm, c[k])) cm |= 1u << k;
    for (; cm; cm &= cm - 1)
      if ((bits_at(kinf, nnz, e + __builtin_ctz(cm), mode) >> 9) < thr) return true;
  }
  return false;
}

// A row of degree <= 32 scanned by kLanes lanes, 32 / kLanes entries each; every
// lane of the group returns whether one of them infects.
template <int kLanes>
__device__ __forceinline__ bool scan_light_group(const int32_t *__restrict__ col,
                                                 const uint32_t *__restrict__ bm, int32_t lo,
                                                 int32_t hi, Key kinf, int64_t nnz, uint32_t thr,
                                                 int mode) {
  constexpr int kEach = kHeavyDeg / kLanes;
  const int lane = threadIdx.x & 63, part = lane & (kLanes - 1);
  int32_t c[kEach];
#pragma unroll
  for (int k = 0; k < kEach; ++k) {
    const int32_t e = lo + part + k * kLanes;
    c[k] = e < hi ? col[e] : -1;
  }
  uint32_t cm = 0;
#pragma unroll
  for (int k = 0; k < kEach; ++k)
    if (c[k] >= 0 && infected(bm, c[k])) cm |= 1u << k;
  bool hit = false;
  for (; cm && !hit; cm &= cm - 1)
    hit = (bits_at(kinf, nnz, lo + part + __builtin_ctz(cm) * kLanes, mode) >> 9) < thr;
  constexpr uint64_t kGroup = (1ull << kLanes) - 1;
  return (__ballot(hit) >> (lane & ~(kLanes - 1)) & kGroup) != 0;
}

// Marks of a row of degree <= 32 by one lane.
__device__ __forceinline__ void mark_light(const int32_t *__restrict__ col,
                                           uint16_t *__restrict__ mark, int32_t e, int32_t hi,
                                           int64_t nnz, uint16_t m) {
  for (; e < hi; e += kRowRound) {
    int32_t c[kRowRound];
    load_row_round(col, e, hi, nnz, c);
#pragma unroll
    for (int k = 0; k < kRowRound; ++k)
      if (c[k] >= 0) mark[c[k]] = m;
  }
}

// Row bounds of item k of a worklist (empty when k is past its end).
__device__ __forceinline__ int2 item_bounds(const SirStep &a, int64_t sub, bool valid, int loc) {
  if (!valid) return make_int2(0, 0);
  const int64_t u = sub + loc;
  return make_int2(a.row_ptr[u], a.row_ptr[u + 1]);
}

__device__ __forceinline__ void mark_heavy(const int32_t *__restrict__ col,
                                           uint16_t *__restrict__ mark,
                                           int64_t lo, int64_t hi, uint16_t m) {
  const int lane = threadIdx.x & 63;
  for (int64_t b = lo; b < hi; b += 8 * 64) {
    int32_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t e = b + k * 64 + lane;
      c[k] = e < hi ? col[e] : -1;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (c[k] >= 0) mark[c[k]] = m;
  }
}

// Push this thread's agents whose bit is set in lmask (light rows, front of
// the list) / hmask (heavy rows, back of the list); agent j of a thread has
// tile index tid * kPerThread + j.  One ballot per (list, j) and one LDS
// atomic per wave and list.
__device__ __forceinline__ void push_items(uint32_t lmask, uint32_t hmask, uint16_t *items,
                                           int32_t *nl, int32_t *nh) {
  const int tid = threadIdx.x, lane = tid & 63;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  uint64_t bl[kPerThread], bh[kPerThread];
  int32_t tl = 0, th = 0;
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    bl[j] = __ballot((lmask >> j) & 1u);
    bh[j] = __ballot((hmask >> j) & 1u);
    tl += (int32_t)__popcll(bl[j]);
    th += (int32_t)__popcll(bh[j]);
  }
  int32_t fl = 0, fh = 0;
  if (lane == 0) {
    if (tl) fl = atomicAdd(nl, tl);
    if (th) fh = atomicAdd(nh, th);
  }
  fl = __shfl(fl, 0);
  fh = __shfl(fh, 0);
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const uint16_t loc = (uint16_t)(tid * kPerThread + j);
    if ((lmask >> j) & 1u) items[fl + __popcll(bl[j] & lt)] = loc;
    if ((hmask >> j) & 1u) items[kTile - 1 - (fh + __popcll(bh[j] & lt))] = loc;
    fl += (int32_t)__popcll(bl[j]);
    fh += (int32_t)__popcll(bh[j]);
  }
}

// The light rows of a worklist by groups of kLanes lanes.
template <int kLanes, int kMode>
__device__ __forceinline__ void scan_light_groups(const SirStep &a,
                                                  const uint32_t *__restrict__ bm, int64_t sub,
                                                  int32_t nl, const uint16_t *items,
                                                  uint8_t *outb, Key kinf) {
  const int32_t k = (int32_t)threadIdx.x / kLanes;  // nl <= kSirThreads / kLanes
  const int loc = k < nl ? (int)items[k] : 0;
  const int2 at = item_bounds(a, sub, k < nl, loc);
  const bool hit =
      scan_light_group<kLanes>(a.col, bm, at.x, at.y, kinf, a.nnz, a.thr_beta, kMode);
  if (hit && (threadIdx.x & (kLanes - 1)) == 0) outb[loc] = 1;
}

// Phase-2 scans of a tile's worklist (heavy rows at its back, light rows at its
// front); a hit marks the agent infected.  Where a tile has few rows, as in
// graphs of some 10,000 agents, the step is bound by the longest chain of
// loads and draws of one lane, so the entries are spread over all lanes: heavy
// rows in units of 64 entries dealt to the wavefronts, four in flight, and up
// to 256 light rows by several lanes each.  20,011 agents x 160 steps: 1,493 us
// a pass against 1,680 with a wavefront a heavy row and a lane a light one (peak
// steps 18.8 -> 14 us); 1M agents x 365 steps 3.11 -> 2.92 ms.
template <int kMode>
__device__ __forceinline__ void scan_items(const SirStep &a, const uint32_t *__restrict__ bm,
                                           int64_t sub, int32_t nl, int32_t nh,
                                           const uint16_t *items, uint8_t *outb, Key kinf) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int kWaves = kSirThreads / 64;
  constexpr int kFlight = 4;
  for (int32_t k0 = 0; k0 < nh; k0 += 64) {
    // lane j holds row k0 + j: its place, bounds and the units up to its end
    const int32_t mine = k0 + lane;
    const int my_loc = mine < nh ? (int)items[kTile - 1 - mine] : 0;
    const int2 my = item_bounds(a, sub, mine < nh, my_loc);
    int32_t ends = (my.y - my.x + 63) >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(ends, off);
      if (lane >= off) ends += y;
    }
    const int32_t units = __builtin_amdgcn_readlane(ends, 63);
    for (int32_t u0 = wave; u0 < units; u0 += kFlight * kWaves) {
      int32_t c[kFlight], e[kFlight];
      int loc[kFlight];
#pragma unroll
      for (int q = 0; q < kFlight; ++q) {
        const int32_t u = u0 + q * kWaves;
        c[q] = -1;
        e[q] = 0;
        loc[q] = 0;
        if (u < units) {  // wave-uniform
          const int j = (int)__popcll(__ballot(ends <= u));
          const int32_t before = j ? __builtin_amdgcn_readlane(ends, j - 1) : 0;
          loc[q] = __builtin_amdgcn_readlane(my_loc, j);
          e[q] = __builtin_amdgcn_readlane(my.x, j) + 64 * (u - before) + lane;
          if (e[q] < __builtin_amdgcn_readlane(my.y, j)) c[q] = a.col[e[q]];
        }
      }
      uint32_t cm = 0, hits = 0;
#pragma unroll
      for (int q = 0; q < kFlight; ++q)
        if (c[q] >= 0 && infected(bm, c[q])) cm |= 1u << q;
      for (; cm; cm &= cm - 1) {
        const int q = __builtin_ctz(cm);
        int32_t at = e[0];
#pragma unroll
        for (int i = 1; i < kFlight; ++i) at = q == i ? e[i] : at;
        if ((bits_at(kinf, a.nnz, at, kMode) >> 9) < a.thr_beta) hits |= 1u << q;
      }
#pragma unroll
      for (int q = 0; q < kFlight; ++q)
        if (__ballot(hits >> q & 1u) && lane == 0) outb[loc[q]] = 1;
    }
  }
  if (nl <= kSirThreads / 16) {
    if (nl > 0) scan_light_groups<16, kMode>(a, bm, sub, nl, items, outb, kinf);
  } else if (nl <= kSirThreads / 4) {
    scan_light_groups<4, kMode>(a, bm, sub, nl, items, outb, kinf);
  } else {
    // a lane each; the next row's bounds load under this one's scan
    int loc = tid < nl ? (int)items[tid] : 0;
    int2 at = item_bounds(a, sub, tid < nl, loc);
    for (int32_t k = tid; k < nl; k += kSirThreads) {
      const int32_t kn = k + kSirThreads;
      const int next_loc = kn < nl ? (int)items[kn] : 0;
      const int2 next = item_bounds(a, sub, kn < nl, next_loc);
      if (scan_light(a.col, bm, at.x, at.y, kinf, a.nnz, a.thr_beta, kMode)) outb[loc] = 1;
      loc = next_loc;
      at = next;
    }
  }
}

// Every exchange between the threads of a block goes through LDS (state, marks
// and bitmaps are never read back by another thread of the block in the same
// step), so its barriers are lds_barrier().
template <bool kLds, int kMode>
__global__ void __launch_bounds__(kSirThreads) k_sir_step(SirStep a) {
  extern __shared__ uint4 lds_bm4[];  // kLds: the bitmap words
  __shared__ __align__(16) uint8_t outb[kTile];
  __shared__ __align__(16) uint16_t items[kTile];
  __shared__ int32_t n_light, n_heavy, m_light, m_heavy;
  __shared__ int32_t cnt[3];
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < 3) cnt[tid] = 0;
  if (a.begun && blockIdx.x == 0 && tid == 0) tell_host(&a.watch[0], a.begun);
  // the first chunk's bounds and the previous step's live flag (one
  // uniform word: no block-wide reduction or barrier) load together
  int64_t c0 = a.chunk_ptr[blockIdx.x], c1 = a.chunk_ptr[blockIdx.x + 1];
  const bool any_inf = a.prev_slots ? a.prev_slots[kLiveFlag] != 0 : true;
  if (!any_inf) {
    // identity step.  Its slots stay zero (the count reduction carries the
    // previous step's counts forward).  The next bitmap B[(t+1)&1] is the
    // infected set after step t-2: empty when step t-2 left no infected agent,
    // so only the first identity step clears its spans.
    if (a.watch && blockIdx.x == 0 && tid == 0) tell_host(&a.watch[1], 1);
    if (!(a.prev2_slots && a.prev2_slots[kLiveFlag] == 0)) {
      for (int32_t c = blockIdx.x; c < a.n_chunks; c += gridDim.x) {
        const int64_t w0 = (int64_t)a.chunk_ptr[c] >> 5;
        const int64_t w1 = c + 1 == a.n_chunks ? a.words : ((int64_t)a.chunk_ptr[c + 1] >> 5);
        for (int64_t w = w0 + tid; w < w1; w += kSirThreads) a.bm_out[w] = 0u;
      }
    }
    return;
  }
  bool staged = false;
  const Key kinf{a.keys[0], a.keys[1]};
  const Key krec{a.keys[2], a.keys[3]};
  const uint16_t new_mark = (uint16_t)(a.t + kMarkHorizon);
  uint32_t c_s = 0, c_i = 0, c_all = 0;  // wave-uniform counts
  uint8_t *bm_out_bytes = reinterpret_cast<uint8_t *>(a.bm_out);
  for (int32_t c = blockIdx.x; c < a.n_chunks; c += gridDim.x) {
    if (c != (int32_t)blockIdx.x) {
      c0 = a.chunk_ptr[c];
      c1 = a.chunk_ptr[c + 1];
    }
    for (int64_t sub = c0; sub < c1; sub += kTile) {
      if (tid == 0) {
        n_light = n_heavy = m_light = m_heavy = 0;
      }
      // phase 1: this thread's 8 consecutive agents v0 .. v0+7 (one 8-byte
      // state load, one 16-byte mark load; chunk starts are 64-aligned)
      const int64_t v0 = sub + (int64_t)tid * kPerThread;
      const int nv = v0 >= c1 ? 0 : (int)(c1 - v0 < kPerThread ? c1 - v0 : kPerThread);
      uint8_t b[kPerThread];
      uint16_t mk[kPerThread];
      if (nv == kPerThread) {
        const uint2 sw = *reinterpret_cast<const uint2 *>(a.state + v0);
        const uint4 mw = *reinterpret_cast<const uint4 *>(a.mark + v0);
        const uint32_t sws[2] = {sw.x, sw.y};
        const uint32_t mws[4] = {mw.x, mw.y, mw.z, mw.w};
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) {
          b[j] = (uint8_t)(sws[j >> 2] >> (8 * (j & 3)));
          mk[j] = (uint16_t)(mws[j >> 1] >> (16 * (j & 1)));
        }
      } else {
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) {
          b[j] = j < nv ? a.state[v0 + j] : (uint8_t)(kHeavyBit | 2);
          mk[j] = j < nv ? a.mark[v0 + j] : (uint16_t)(a.t + 0x8000u);
        }
      }
      uint32_t lmask = 0, hmask = 0, imask = 0;
      uint32_t ob[2] = {0u, 0u};
#pragma unroll
      for (int j = 0; j < kPerThread; ++j) {
        const uint8_t s = b[j] & 3;
        ob[j >> 2] |= (uint32_t)s << (8 * (j & 3));
        if (s == 1) imask |= 1u << j;
        if (s == 0 && at_risk(mk[j], a.t)) {
          if (b[j] & kHeavyBit) hmask |= 1u << j;
          else lmask |= 1u << j;
        }
      }
      // recoveries: a thread's own, one after the other, or in a small tile one
      // a thread after the barrier
      const bool small = c1 - sub <= kSirThreads;  // block-uniform
      for (uint32_t m = small ? 0u : imask; m; m &= m - 1) {
        const int j = __builtin_ctz(m);
        if ((bits_at(krec, a.n, v0 + j, kMode) >> 9) < a.thr_gamma)
          ob[j >> 2] ^= 3u << (8 * (j & 3));  // I (1) -> R (2)
      }
      *reinterpret_cast<uint2 *>(outb + tid * kPerThread) = make_uint2(ob[0], ob[1]);
      lds_barrier();  // counters reset before any push
      push_items(lmask, hmask, items, &n_light, &n_heavy);
      if (small && sub + tid < c1 && outb[tid] == 1 &&
          (bits_at(krec, a.n, sub + tid, kMode) >> 9) < a.thr_gamma)
        outb[tid] = 2;
      lds_barrier();
      // phase 2: scans against the LDS copy of the bitmap when the tile has
      // enough rows, else the global one
      // (block-uniform: a tile with no row to scan writes no other thread's
      // outb byte, so it needs no barrier before phase 3)
      {
        const int32_t nl = n_light, nh = n_heavy;
        if (nl + nh > 0) {
          if constexpr (kLds) {
            if (!staged && nl + nh >= kStageItems) {
              const uint4 *src = reinterpret_cast<const uint4 *>(a.bm_in);
              for (int64_t i = tid; i < (a.words >> 2); i += kSirThreads) lds_bm4[i] = src[i];
              staged = true;
              lds_barrier();
            }
          }
          if (kLds && staged)
            scan_items<kMode>(a, reinterpret_cast<const uint32_t *>(lds_bm4), sub, nl, nh,
                              items, outb, kinf);
          else
            scan_items<kMode>(a, a.bm_in, sub, nl, nh, items, outb, kinf);
          lds_barrier();
        }
      }
      // phase 3: outputs (one 8-byte state store when anything changed), the
      // next bitmap (one byte = these 8 agents), counts, the mark worklist
      const uint2 rw = *reinterpret_cast<const uint2 *>(outb + tid * kPerThread);
      const uint32_t rws[2] = {rw.x, rw.y};
      lmask = 0;
      hmask = 0;
      uint32_t ibits = 0, sbits = 0, changed = 0;
      uint32_t nw[2] = {0u, 0u};
#pragma unroll
      for (int j = 0; j < kPerThread; ++j) {
        const uint8_t s = b[j] & 3;
        const uint8_t r = (uint8_t)(rws[j >> 2] >> (8 * (j & 3)));
        nw[j >> 2] |= (uint32_t)(r | (b[j] & kHeavyBit)) << (8 * (j & 3));
        if (j < nv) {
          changed |= r != s;
          ibits |= (uint32_t)(r == 1) << j;
          sbits |= (uint32_t)(r == 0) << j;
          const bool refresh = ((a.t + (uint32_t)(v0 + j)) % kMarkHorizon) == 0;
          if (r == 1 && (s == 0 || refresh)) {
            if (b[j] & kHeavyBit) hmask |= 1u << j;
            else lmask |= 1u << j;
          }
        }
      }
      if (changed) {
        if (nv == kPerThread) {
          *reinterpret_cast<uint2 *>(a.state + v0) = make_uint2(nw[0], nw[1]);
        } else {
#pragma unroll
          for (int j = 0; j < kPerThread; ++j)
            if (j < nv) a.state[v0 + j] = (uint8_t)(nw[j >> 2] >> (8 * (j & 3)));
        }
      }
      if (nv > 0) bm_out_bytes[v0 >> 3] = (uint8_t)ibits;
      c_s += (uint32_t)__popc(sbits);
      c_i += (uint32_t)__popc(ibits);
      c_all += (uint32_t)nv;
      // the scan worklist is dead after the barrier above; reuse it for marks
      push_items(lmask, hmask, items, &m_light, &m_heavy);
      lds_barrier();
      // phase 4: marks of newly infected agents and periodic refreshes
      // (block-uniform: with none, no thread reads the worklist or its
      // counters, and the next tile's reset only rewrites zeros)
      {
        const int32_t nl = m_light, nh = m_heavy;
        if (nl + nh > 0) {
          const int wave = tid >> 6;
          for (int32_t k = wave; k < nh; k += kSirThreads / 64) {
            const int64_t u = sub + items[kTile - 1 - k];
            mark_heavy(a.col, a.mark, a.row_ptr[u], a.row_ptr[u + 1], new_mark);
          }
          for (int32_t k = tid; k < nl; k += kSirThreads) {
            const int2 at = item_bounds(a, sub, true, items[k]);
            mark_light(a.col, a.mark, at.x, at.y, a.nnz, new_mark);
          }
          lds_barrier();
        }
      }
    }
  }
  // block counts: per-thread counts -> wave sums -> LDS -> one atomic per class
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    c_s += __shfl_xor(c_s, off);
    c_i += __shfl_xor(c_i, off);
    c_all += __shfl_xor(c_all, off);
  }
  if (lane == 0) {
    atomicAdd(&cnt[0], (int32_t)c_s);
    atomicAdd(&cnt[1], (int32_t)c_i);
    atomicAdd(&cnt[2], (int32_t)(c_all - c_s - c_i));
  }
  lds_barrier();
  if (tid < 3 && cnt[tid]) atomicAdd(&a.slots[(blockIdx.x % kSlots) * 3 + tid], cnt[tid]);
  if (tid == 1 && cnt[1]) a.slots[kLiveFlag] = 1;
}

// counts[t][k] = sum over the count slots of slots[t][s][k]; an identity
// step leaves its slots zero (S + I + R = n > 0 for any computed step), which
// this pass records in the flag slot's spare word for the carry pass
constexpr int kComputedMark = kSlots * 3;

__global__ void k_sir_reduce_slots(int32_t *__restrict__ slots, int64_t steps,
                                   int32_t *__restrict__ counts) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= steps * 3) return;
  const int64_t t = i / 3, k = i - t * 3;
  const int32_t *p = slots + t * kStride + k;
  int32_t s = 0;
  for (int j = 0; j < kSlots; ++j) s += p[j * 3];
  counts[i] = s;
  if (k == 0) {
    int32_t tot = 0;
    for (int j = 0; j < kSlots * 3; ++j) tot |= slots[t * kStride + j];
    slots[t * kStride + kComputedMark] = tot != 0;
  }
}

// Identity steps form a suffix of a run (no infected agent, no new
// infection): counts[t] = counts[t_a - 1] for t >= t_a, the first identity
// step, found by binary search over the computed marks.
__global__ void k_sir_carry_counts(const int32_t *__restrict__ slots, int64_t steps,
                                   int32_t *__restrict__ counts) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= steps * 3) return;
  const int64_t t = i / 3, k = i - t * 3;
  if (slots[t * kStride + kComputedMark]) return;
  int64_t lo = 0, hi = t;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (slots[mid * kStride + kComputedMark])
      lo = mid + 1;
    else
      hi = mid;
  }
  counts[i] = lo > 0 ? counts[(lo - 1) * 3 + k] : 0;
}

__global__ void k_fill_i32(int32_t *__restrict__ p, int64_t n, int32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// state[v] = S with the heavy-row flag.
__global__ void k_sir_init_state(int64_t n, const int32_t *__restrict__ row_ptr,
                                 uint8_t *__restrict__ state) {
  int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n) state[v] = (row_ptr[v + 1] - row_ptr[v] > kHeavyDeg) ? kHeavyBit : 0;
}

__global__ void k_sir_seed(const int32_t *__restrict__ perm, int64_t n0,
                           uint8_t *__restrict__ state) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n0) state[perm[i]] = (state[perm[i]] & kHeavyBit) | 1;
}

__global__ void k_fill_u16(uint16_t *__restrict__ p, int64_t n, uint16_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Initial marks: every infected agent marks its neighbours with `m`.
__global__ void k_sir_mark_infected(int64_t n, const int32_t *__restrict__ row_ptr,
                                    const int32_t *__restrict__ col,
                                    const uint8_t *__restrict__ state,
                                    uint16_t *__restrict__ mark, uint16_t m) {
  int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n || (state[v] & 3) != 1) return;
  for (int64_t e = row_ptr[v]; e < row_ptr[v + 1]; ++e) mark[col[e]] = m;
}

// bitmap word w = infected bits of agents 32w .. 32w+31
__global__ void k_sir_bitmap(int64_t n, const uint8_t *__restrict__ state,
                             int64_t words, uint32_t *__restrict__ bm) {
  int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= words) return;
  uint32_t x = 0;
  for (int k = 0; k < 32; ++k) {
    const int64_t v = w * 32 + k;
    if (v < n && (state[v] & 3) == 1) x |= 1u << k;
  }
  bm[w] = x;
}

__global__ void k_mask_state(const uint8_t *__restrict__ in, int64_t n,
                             uint8_t *__restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i] & 3;
}

inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

inline int64_t bitmap_words(int64_t n) { return ((n + 127) / 128) * 4; }

int check_graph(const abm_sir_graph *g, const char *who) {
  if (!g || g->n <= 0 || g->n >= (1ll << 31) - 64 || g->nnz < 0 ||
      g->nnz >= (1ll << 31) - 64 || g->n_chunks < 1 || g->n_chunks > g->n ||
      !g->row_ptr || (g->nnz && !g->col) || !g->chunk_ptr) {
    set_error(std::string(who) + ": bad graph descriptor");
    return kErrInvalid;
  }
  return kOk;
}

// The chunk table the step kernel assumes: chunk_ptr[0] = 0, chunk_ptr
// [n_chunks] = n, ascending, every inner boundary a multiple of kChunkAlign
// (each bitmap byte and 8-agent state word then has one owning block) and no
// chunk longer than one tile.  Read back once per instance set-up.
int check_chunks(const abm_sir_graph *g, hipStream_t s) {
  std::vector<int32_t> cp((size_t)g->n_chunks + 1);
  ABM_CHECK_HIP(hipMemcpyAsync(cp.data(), g->chunk_ptr, cp.size() * sizeof(int32_t),
                               hipMemcpyDeviceToHost, s));
  ABM_CHECK_HIP(hipStreamSynchronize(s));
  bool ok = cp.front() == 0 && cp.back() == g->n;
  for (size_t i = 1; ok && i < cp.size(); ++i) {
    ok = cp[i] > cp[i - 1] && cp[i] - cp[i - 1] <= kTile;
    if (i + 1 < cp.size()) ok = ok && cp[i] % kChunkAlign == 0;
  }
  if (!ok) {
    set_error("abm_sir_seed: chunk_ptr must run from 0 to n, ascending, with inner boundaries "
              "multiples of 64 and chunks of at most 8192 agents (abm_node_chunks with "
              "abm_sir_chunk_params)");
    return kErrInvalid;
  }
  return kOk;
}

// The bitmap-staging kernels need more than 64 KB of dynamic LDS: the limit
// is raised once per device (under a lock; each device keeps its own
// function attributes).
constexpr int kMaxDevices = 64;
std::mutex g_lds_attr_mu;
bool g_lds_attr_set[kMaxDevices];

int sir_lds_attr() {
  int dev = -1;
  ABM_CHECK_HIP(hipGetDevice(&dev));
  ABM_REQUIRE(dev >= 0 && dev < kMaxDevices, "sir: device index out of range");
  std::lock_guard<std::mutex> lock(g_lds_attr_mu);
  if (!g_lds_attr_set[dev]) {
    for (const void *k : {(const void *)k_sir_step<true, kModePartitionable>,
                          (const void *)k_sir_step<true, kModeOriginal>})
      ABM_CHECK_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)(kLdsBitmapWords * 4)));
    g_lds_attr_set[dev] = true;
  }
  return kOk;
}

int check_aligned(const void *p, uintptr_t bytes, const char *who, const char *what) {
  if (((uintptr_t)p & (bytes - 1)) != 0) {
    set_error(std::string(who) + ": " + what + " must be " + std::to_string(bytes) +
              "-byte aligned");
    return kErrInvalid;
  }
  return kOk;
}

int check_buffers(const uint8_t *state, const uint16_t *mark, const uint32_t *b0,
                  const uint32_t *b1, const char *who) {
  if (int rc = check_aligned(state, 8, who, "state")) return rc;
  if (int rc = check_aligned(mark, 16, who, "mark")) return rc;
  if (int rc = check_aligned(b0, 16, who, "bitmap")) return rc;
  return check_aligned(b1, 16, who, "bitmap");
}

int launch_step(const abm_sir_graph *g, uint8_t *state, uint16_t *mark,
                const uint32_t *bm_in, uint32_t *bm_out, uint32_t t,
                const uint32_t *keys4, uint32_t tb, uint32_t tg, int mode,
                const int32_t *prev_slots, const int32_t *prev2_slots, int32_t *slots,
                int32_t *watch, int32_t begun, hipStream_t s) {
  SirStep a;
  a.watch = watch;
  a.begun = begun;
  a.n = g->n;
  a.nnz = g->nnz;
  a.row_ptr = g->row_ptr;
  a.col = g->col;
  a.chunk_ptr = g->chunk_ptr;
  a.n_chunks = (int32_t)g->n_chunks;
  a.state = state;
  a.mark = mark;
  a.bm_in = bm_in;
  a.bm_out = bm_out;
  a.words = bitmap_words(g->n);
  a.t = t;
  a.prev_slots = prev_slots;
  a.prev2_slots = prev2_slots;
  a.keys = keys4;
  a.thr_beta = tb;
  a.thr_gamma = tg;
  a.slots = slots;
  const unsigned blocks = (unsigned)(g->n_chunks < kSirBlocks ? g->n_chunks : kSirBlocks);
  // one instantiation per stream layout: each carries one copy of the draw
  const bool part = mode == kModePartitionable;
  if (a.words <= kLdsBitmapWords) {
    auto *kp = k_sir_step<true, kModePartitionable>;
    auto *ko = k_sir_step<true, kModeOriginal>;
    if (int rc = sir_lds_attr()) return rc;
    hipLaunchKernelGGL(part ? kp : ko, dim3(blocks), dim3(kSirThreads), (size_t)a.words * 4,
                       s, a);
  } else {
    auto *kg = part ? k_sir_step<false, kModePartitionable> : k_sir_step<false, kModeOriginal>;
    hipLaunchKernelGGL(kg, dim3(blocks), dim3(kSirThreads), 0, s, a);
  }
  return kOk;
}

// A watched run learns from the step kernels themselves how far it is (a store
// to host memory at a step's start, no launch or copy of its own).  The store
// costs its step about 1 us at the end, so only every kWatchEvery-th step
// tells; the host launches kWatchEvery steps once the step as many before them
// has begun, and up to twice as many identity steps, 2 us each, follow the last
// infection.  1M agents x 365 steps: 3.34 ms a pass when every step tells,
// 3.11 when each eighth does, 3.25 without a watch.
constexpr int32_t kWatchEvery = 8;

// The steps of a run; with watch, launching stops once a step was the identity:
// so is every later one, and the count reduction fills in their zeroed slots as
// if they had been launched.
int sir_run(const char *who, const abm_sir_graph *g, uint8_t *state, uint16_t *mark,
            uint32_t *bitmaps, uint32_t t0, const uint32_t *keys, int32_t steps, float beta,
            float gamma, int mode, int32_t *slots, int32_t *counts, int32_t *watch,
            int32_t *launched, hipStream_t s) {
  if (int rc = check_graph(g, who)) return rc;
  if (!(state && mark && bitmaps && keys && slots && counts)) {
    set_error(std::string(who) + ": null buffer");
    return kErrInvalid;
  }
  if (!(steps >= 0 && (mode == 0 || mode == 1))) {
    set_error(std::string(who) + ": bad steps or mode");
    return kErrInvalid;
  }
  if (int rc = check_buffers(state, mark, bitmaps, bitmaps + bitmap_words(g->n), who)) return rc;
  if (steps == 0) return kOk;
  const uint32_t tb = unit_threshold(beta), tg = unit_threshold(gamma);
  const int64_t words = bitmap_words(g->n);
  const int64_t ns = (int64_t)steps * kStride;
  // too short to stop: no step tells (4 steps after the last infection: 66 us
  // with the stores, 62 without)
  if (steps <= 2 * kWatchEvery) watch = nullptr;
  if (watch) clear_watch(watch);
  hipLaunchKernelGGL(k_fill_i32, dim3(blocks_for(ns, 256)), dim3(256), 0, s,
                     slots, ns, 0);
  uint32_t *bm[2] = {bitmaps, bitmaps + words};
  int32_t t = 0;
  for (; t < steps; ++t) {
    const bool tells = watch && t % kWatchEvery == 0;
    if (tells && t >= 2 * kWatchEvery) {
      bool settled = false;
      if (int rc = wait_begun(watch, t + 1 - kWatchEvery, s, who, &settled)) return rc;
      if (settled) break;
    }
    if (int rc = launch_step(g, state, mark, bm[t & 1], bm[(t + 1) & 1],
                             t0 + (uint32_t)t, keys + 4 * (int64_t)t, tb, tg, mode,
                             t ? slots + (int64_t)(t - 1) * kStride : nullptr,
                             t > 1 ? slots + (int64_t)(t - 2) * kStride : nullptr,
                             slots + (int64_t)t * kStride, watch, tells ? t + 1 : 0, s))
      return rc;
  }
  hipLaunchKernelGGL(k_sir_reduce_slots, dim3(blocks_for(3 * (int64_t)steps, 256)),
                     dim3(256), 0, s, slots, (int64_t)steps, counts);
  hipLaunchKernelGGL(k_sir_carry_counts, dim3(blocks_for(3 * (int64_t)steps, 256)),
                     dim3(256), 0, s, (const int32_t *)slots, (int64_t)steps, counts);
  if (t & 1)
    ABM_CHECK_HIP(hipMemcpyAsync(bm[0], bm[1], (size_t)words * 4,
                                 hipMemcpyDeviceToDevice, s));
  if (launched) *launched = t;
  ABM_LAUNCH_CHECK(who);
  return kOk;
}

}  // namespace abm

using namespace abm;

extern "C" {

int abm_fill_i32(int32_t *p, int64_t n, int32_t v, void *stream) {
  ABM_REQUIRE(n >= 0, "abm_fill_i32: n must be >= 0");
  if (n == 0) return kOk;
  hipLaunchKernelGGL(k_fill_i32, dim3(blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, p, n, v);
  ABM_LAUNCH_CHECK("abm_fill_i32");
  return kOk;
}

uint32_t abm_unit_threshold(float p) { return unit_threshold(p); }

int abm_sir_slots(void) { return kStepSlots; }

int64_t abm_sir_bitmap_words(int64_t n) { return n > 0 ? bitmap_words(n) : 0; }

int abm_sir_chunk_params(int32_t *align, int64_t *node_cost, int32_t *heavy_deg,
                         int64_t *heavy_cost, int32_t *chunks_per_block, int32_t *blocks,
                         int32_t *max_nodes) {
  if (align) *align = kChunkAlign;
  if (heavy_deg) *heavy_deg = kHeavyDeg;
  if (heavy_cost) *heavy_cost = kChunkHeavyCost;
  if (max_nodes) *max_nodes = kTile;
  if (node_cost) *node_cost = kChunkNodeCost;
  if (chunks_per_block) *chunks_per_block = kChunksPerBlock;
  if (blocks) *blocks = kSirBlocks;
  return kOk;
}

int abm_sir_seed(const abm_sir_graph *g, const int32_t *perm, int64_t n0,
                 uint8_t *state, uint16_t *mark, uint32_t *bitmap, uint32_t t0,
                 void *stream) {
  if (int rc = check_graph(g, "abm_sir_seed")) return rc;
  ABM_REQUIRE(state && mark && bitmap && n0 >= 0 && n0 <= g->n && (n0 == 0 || perm),
              "abm_sir_seed: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  if (int rc = check_chunks(g, s)) return rc;
  // the per-device launch set-up, here rather than inside a captured run
  if (int rc = sir_lds_attr()) return rc;
  const int64_t n = g->n, words = bitmap_words(n);
  hipLaunchKernelGGL(k_sir_init_state, dim3(blocks_for(n, 256)), dim3(256), 0,
                     s, n, g->row_ptr, state);
  if (n0 > 0)
    hipLaunchKernelGGL(k_sir_seed, dim3(blocks_for(n0, 256)), dim3(256), 0, s,
                       perm, n0, state);
  hipLaunchKernelGGL(k_fill_u16, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                     mark, n, (uint16_t)(t0 + 0x8000u));
  hipLaunchKernelGGL(k_sir_mark_infected, dim3(blocks_for(n, 256)), dim3(256), 0,
                     s, n, g->row_ptr, g->col, state, mark,
                     (uint16_t)(t0 + kMarkHorizon));
  hipLaunchKernelGGL(k_sir_bitmap, dim3(blocks_for(words, 256)), dim3(256), 0,
                     s, n, state, words, bitmap);
  ABM_LAUNCH_CHECK("abm_sir_seed");
  return kOk;
}

int abm_sir_run(const abm_sir_graph *g, uint8_t *state, uint16_t *mark,
                uint32_t *bitmaps, uint32_t t0, const uint32_t *keys,
                int32_t steps, float beta, float gamma, int mode, int32_t *slots,
                int32_t *counts, void *stream) {
  return sir_run("abm_sir_run", g, state, mark, bitmaps, t0, keys, steps, beta, gamma, mode, slots,
                 counts, nullptr, nullptr, (hipStream_t)stream);
}

int abm_sir_run_watched(const abm_sir_graph *g, uint8_t *state, uint16_t *mark,
                        uint32_t *bitmaps, uint32_t t0, const uint32_t *keys, int32_t steps,
                        float beta, float gamma, int mode, int32_t *slots, int32_t *counts,
                        int32_t *watch, int32_t *launched, void *stream) {
  ABM_REQUIRE(watch && launched, "abm_sir_run_watched: null buffer");
  *launched = 0;
  return sir_run("abm_sir_run_watched", g, state, mark, bitmaps, t0, keys, steps, beta, gamma,
                 mode, slots, counts, watch, launched, (hipStream_t)stream);
}

int abm_sir_step(const abm_sir_graph *g, uint8_t *state, uint16_t *mark,
                 const uint32_t *bm_in, uint32_t *bm_out, uint32_t t,
                 const uint32_t *keys4, float beta, float gamma, int mode,
                 const int32_t *prev_slots, int32_t *slots, void *stream) {
  if (int rc = check_graph(g, "abm_sir_step")) return rc;
  ABM_REQUIRE(state && mark && bm_in && bm_out && keys4 && slots && bm_in != bm_out &&
                  (mode == 0 || mode == 1),
              "abm_sir_step: bad argument");
  if (int rc = check_buffers(state, mark, bm_in, bm_out, "abm_sir_step")) return rc;
  if (int rc = launch_step(g, state, mark, bm_in, bm_out, t, keys4, unit_threshold(beta),
                           unit_threshold(gamma), mode, prev_slots, nullptr, slots, nullptr, 0,
                           (hipStream_t)stream))
    return rc;
  ABM_LAUNCH_CHECK("abm_sir_step");
  return kOk;
}

int abm_sir_reduce_counts(int32_t *slots, int32_t steps, int32_t *counts, void *stream) {
  ABM_REQUIRE(slots && counts && steps >= 0, "abm_sir_reduce_counts: bad args");
  if (steps == 0) return kOk;
  hipLaunchKernelGGL(k_sir_reduce_slots, dim3(blocks_for(3 * (int64_t)steps, 256)),
                     dim3(256), 0, (hipStream_t)stream, slots, (int64_t)steps,
                     counts);
  hipLaunchKernelGGL(k_sir_carry_counts, dim3(blocks_for(3 * (int64_t)steps, 256)),
                     dim3(256), 0, (hipStream_t)stream, (const int32_t *)slots,
                     (int64_t)steps, counts);
  ABM_LAUNCH_CHECK("abm_sir_reduce_counts");
  return kOk;
}

int abm_sir_states(const uint8_t *state, int64_t n, uint8_t *out, void *stream) {
  ABM_REQUIRE(state && out && n >= 0, "abm_sir_states: bad args");
  if (n == 0) return kOk;
  hipLaunchKernelGGL(k_mask_state, dim3(blocks_for(n, 256)), dim3(256), 0,
                     (hipStream_t)stream, state, n, out);
  ABM_LAUNCH_CHECK("abm_sir_states");
  return kOk;
}

}  // extern "C"
