// wealth.hip -- wealth-exchange random walk: batches of instances, and one large
// instance over the whole GPU.
//
// Program (reference API, jaxabm/model.py:118-216, jaxabm/agent.py:92-177):
//  init   agent keys = split(init_key, n); kx, ky = split(agent_key);
//         x = uniform(kx), y = uniform(ky), wealth = 1
//  step   agent phase (agent keys = split(ck, n)): k1, k2 = split(agent_key);
//           x = mod(x + 0.01 * normal(k1), 1), y = mod(y + 0.01 * normal(k2), 1)
//         env phase (uk): t = randint(uk, (n,), 0, n-1); t += (t >= i);
//           give = wealth > 0; wealth += bincount(t, give) - give
//  record mean(wealth) and Gini (examples/models/advanced_economic_model.py:
//         1798-1811): x = sort(wealth); S = sum(i * x_i) and T = sum(x) in
//         int32; G = f32(2 S) / f32(n T) - f32((n+1)/n) if T > 1e-6.
//
// The sort is replaced by a histogram over wealth values: with c_w agents of
// wealth w and b_w agents below, their ranks sum to c_w * b_w + c_w(c_w+1)/2,
// so S = sum_w w * ranksum_w (mod 2^32, the int32 wrap of the reference).
// Scatter-adds are integer atomics (exact, order-free).
//
// A run with a draw buffer (abm_wealth_run_batch, draws != NULL) is split by
// what depends on what.  The draws depend on nothing, so a grid-wide kernel
// makes all of them first.  The walk depends on its own agent's draws only,
// and a record only on its step's wealth.  What is left as a serial chain over
// the steps is the exchange itself, and that alone runs step after step in
// one workgroup (k_wealth_exchange), leaving every step's wealth in the draw
// buffer; beside it other workgroups walk the positions, and after it the
// records of all steps are taken at once, one workgroup per step
// (k_wealth_records).
// Without a draw buffer, or above the size the exchange keeps in LDS, one
// workgroup runs everything: every phase boundary is a workgroup barrier, and
// an instance of up to kWealthLdsAgents agents keeps its arrays in LDS
// (20 bytes per agent), a larger one on its global buffers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#define ABM_STRAIGHT_DRAWS
#include "common.hpp"
#include "jaxabm_amd.h"

namespace abm {

constexpr int kWealthThreads = 1024;
// LDS per resident agent: x, y, wealth, increment, histogram bin
constexpr int64_t kWealthLdsBytesPerAgent = 20;
constexpr int64_t kWealthLdsAgents = 8000;  // 160,020 bytes with the extra bin

__device__ __forceinline__ uint32_t block_sum_u32(uint32_t v, uint32_t *red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (lane == 0) red[wave] = v;
  __syncthreads();
  uint32_t s = 0;
  if (threadIdx.x < 64) {
    s = threadIdx.x < (blockDim.x >> 6) ? red[threadIdx.x] : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  }
  __syncthreads();
  return s;  // valid in wave 0
}

// The draws of agent i at one step (ck: the collection key; kk1, kk2 =
// split(uk), the same for every agent): the position increments 0.01 * normal
// (rounded as the reference's product), and the exchange target.
struct WealthWalk {
  float mdx, mdy;
};

__device__ __forceinline__ WealthWalk wealth_walk(Key ck, int64_t n, int64_t i, int mode) {
  Key k1, k2;
  split2(split_at(ck, n, i, mode), k1, k2, mode);
  WealthWalk d;
  d.mdx = 0.01f * normal_from_bits(bits_scalar(k1, mode));
  d.mdy = 0.01f * normal_from_bits(bits_scalar(k2, mode));
  return d;
}

__device__ __forceinline__ uint32_t wealth_target(Key kk1, Key kk2, int64_t n, int64_t i,
                                                  int mode) {
  const uint32_t span = n > 1 ? (uint32_t)(n - 1) : 1u;
  uint32_t ti = randint_offset(bits_at(kk1, n, i, mode), bits_at(kk2, n, i, mode), span);
  return ti + (ti >= (uint32_t)i ? 1u : 0u);
}

__device__ __forceinline__ Key collection_key(const uint32_t *keys, int32_t t) {
  return Key{keys[4 * t + 0], keys[4 * t + 1]};
}

__device__ __forceinline__ void target_keys(const uint32_t *keys, int32_t t, Key &kk1, Key &kk2,
                                            int mode) {
  split2(Key{keys[4 * t + 2], keys[4 * t + 3]}, kk1, kk2, mode);
}

// Every draw of a run, grid-wide, into draws[steps][3][n] (mdx, mdy bits,
// target): none depends on the state.  Workgroups take tiles of one step and
// kDrawThreads agents, so the step and its keys are uniform.
constexpr int kDrawThreads = 256;

template <int kMode>
__global__ void __launch_bounds__(kDrawThreads)
    k_wealth_draws(const abm_wealth_inst *__restrict__ insts) {
  const abm_wealth_inst in = insts[blockIdx.y];
  if (!in.draws) return;
  const int64_t n = in.n;
  const int64_t per = (n + kDrawThreads - 1) / kDrawThreads;
  for (int64_t q = blockIdx.x; q < (int64_t)in.steps * per; q += gridDim.x) {
    const int32_t t = (int32_t)(q / per);
    const int64_t i = (q - (int64_t)t * per) * kDrawThreads + threadIdx.x;
    if (i >= n) continue;
    Key kk1, kk2;
    target_keys(in.keys, t, kk1, kk2, kMode);
    const WealthWalk d = wealth_walk(collection_key(in.keys, t), n, i, kMode);
    const GlobalPtr<uint32_t> row = as_global(in.draws) + (int64_t)t * 3 * n;
    row[i] = __float_as_uint(d.mdx);
    row[n + i] = __float_as_uint(d.mdy);
    row[2 * n + i] = wealth_target(kk1, kk2, n, i, kMode);
  }
}

// Mean and Gini of a step from its total T and rank sum S.
__device__ __forceinline__ void wealth_write_record(const abm_wealth_inst &in, int32_t t,
                                                    uint32_t T, uint32_t S) {
  const int64_t n = in.n;
  in.mean_out[t] = (float)(int32_t)T / (float)n;
  const int32_t Ti = (int32_t)T;
  float g = 0.0f;
  if ((float)Ti > 1e-6f) {
    const int32_t num = (int32_t)(2u * S);
    const int32_t den = (int32_t)((uint32_t)n * T);
    const float q = (float)num / (float)den;
    const float cst = (float)((double)(n + 1) / (double)n);
    g = q - cst;
  }
  in.gini_out[t] = g;
}

// S = sum_w w * (c_w b_w + c_w (c_w + 1) / 2): chunked exclusive scan of the
// histogram, one bin per thread per chunk, until all n agents are counted
// (which covers every nonzero bin); the bins are cleared.  Valid in thread 0.
__device__ __forceinline__ uint32_t wealth_rank_sum(int32_t *hist, int64_t n, uint32_t *red,
                                                    uint32_t &carry) {
  const int tid = threadIdx.x;
  if (tid == 0) carry = 0;
  __syncthreads();
  uint32_t S_part = 0;
  for (int64_t base = 0; base <= n; base += kWealthThreads) {
    const int64_t w = base + tid;
    const uint32_t c = w <= n ? (uint32_t)hist[w] : 0u;
    // inclusive wave scan of c, then across waves
    uint32_t inc = c;
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off);
      if (lane >= off) inc += y;
    }
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    uint32_t wave_off = 0;
    for (int q = 0; q < wave; ++q) wave_off += red[q];
    const uint32_t before = carry + wave_off + inc - c;
    if (c) {
      const uint64_t ranksum = (uint64_t)c * before + (uint64_t)c * (c + 1) / 2;
      S_part += (uint32_t)w * (uint32_t)ranksum;
      hist[w] = 0;
    }
    __syncthreads();
    if (tid == kWealthThreads - 1) carry = before + c;
    __syncthreads();
    if ((int64_t)carry >= n) break;  // block-uniform
  }
  return block_sum_u32(S_part, red);
}

// The whole run of one instance by one workgroup on the arrays x, y, w
// (state), inc and hist (zero on entry, left zero) -- global buffers or their
// LDS copies.
__device__ __forceinline__ void wealth_steps(const abm_wealth_inst &in, float *gx, float *gy,
                                             int32_t *gw, int32_t *ginc, int32_t *ghist,
                                             uint32_t *red, uint32_t &carry, int mode) {
  const int64_t n = in.n;
  const int tid = threadIdx.x;
  for (int32_t t = 0; t < in.steps; ++t) {
    // agent phase + exchange targets
    for (int64_t i = tid; i < n; i += kWealthThreads) {
      WealthWalk d;
      uint32_t target;
      if (in.draws) {
        const uint32_t *row = in.draws + (int64_t)t * 3 * n;
        d.mdx = __uint_as_float(row[i]);
        d.mdy = __uint_as_float(row[n + i]);
        target = row[2 * n + i];
      } else {
        Key kk1, kk2;
        target_keys(in.keys, t, kk1, kk2, mode);
        target = wealth_target(kk1, kk2, n, i, mode);
        d = wealth_walk(collection_key(in.keys, t), n, i, mode);
      }
      gx[i] = mod1(gx[i] + d.mdx);
      gy[i] = mod1(gy[i] + d.mdy);
      if (gw[i] > 0) atomicAdd(&ginc[target], 1);
    }
    __syncthreads();
    // apply the exchange, histogram of wealth values
    uint32_t total = 0;
    for (int64_t i = tid; i < n; i += kWealthThreads) {
      const int32_t w0 = gw[i];
      const int32_t wi = w0 - (w0 > 0 ? 1 : 0) + ginc[i];
      gw[i] = wi;
      ginc[i] = 0;
      atomicAdd(&ghist[wi], 1);  // 0 <= wi <= n: wealth is conserved
      total += (uint32_t)wi;
    }
    const uint32_t T = block_sum_u32(total, red);
    __syncthreads();
    const uint32_t S = wealth_rank_sum(ghist, n, red, carry);
    if (tid == 0) wealth_write_record(in, t, T, S);
    __syncthreads();
  }
}

// ---- runs with a draw buffer: exchange chain, walk and records apart

// Instances the exchange kernel takes: two LDS arrays of increments, 32-bit up
// to 20 agents a thread, and two agents per word above (a step gives an agent
// at most n - 1 units, so neither half overflows), within 160 KB.
constexpr int64_t kExchangeAgents = 40000;

__host__ __device__ inline bool wealth_split_run(const abm_wealth_inst &in, int64_t cap) {
  return in.draws != nullptr && in.n <= cap;
}

// Words of one increment array: every thread's A agents, or pairs of them.
constexpr int32_t exchange_words(int A, bool packed) {
  return A * kWealthThreads / (packed ? 2 : 1);
}

// Steps ahead that a thread loads its A agents' targets: a step of few agents
// takes less time than a memory round trip.
constexpr int exchange_ahead(int A) { return A <= 2 ? 8 : A <= 8 ? 4 : A <= 16 ? 2 : 1; }

// The exchange chain of one instance by one workgroup: thread t keeps the
// wealth of agents t, t + 1024, .. (A of them) in registers, and a step is one
// LDS atomic per giver, one barrier, and the increments read and cleared
// (alternating arrays, so that one barrier a step is enough).  The wealth
// after step t replaces the step's targets in the draw buffer.
//
// No global access of a step is in a branch: a wait for one load counts the
// accesses issued after it, and a branch around any of them makes that a wait
// for all, a memory round trip in every step (5,003 agents: 1.83 us a step,
// 0.63 this way).  So the rows are accessed as raw buffers of n words, where
// an absent agent's load gives 0 and its store is dropped by the bounds check.
using RowBuffer = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ RowBuffer row_buffer(void *p, int32_t n) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, 4 * n, 0x00020000);
}

template <int A, bool kPacked>
__device__ __forceinline__ void exchange_steps(const abm_wealth_inst &in, uint32_t *lds_inc) {
  constexpr int P = exchange_ahead(A);
  constexpr int32_t words = exchange_words(A, kPacked);
  const uint32_t tid = threadIdx.x;
  const int32_t n = (int32_t)in.n, steps = in.steps;
  const int64_t row = 3 * (int64_t)n;
  uint32_t *targets = in.draws + 2 * (int64_t)n;
  auto load = [&](RowBuffer b, int a) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b, 4 * (tid + a * kWealthThreads), 0, 0);
  };
  auto store = [&](RowBuffer b, int a, uint32_t v) {
    __builtin_amdgcn_raw_buffer_store_b32(v, b, 4 * (tid + a * kWealthThreads), 0, 0);
  };
  uint32_t w[A], target[P][A];
  {
    const RowBuffer wealth = row_buffer(in.w, n);
#pragma unroll
    for (int a = 0; a < A; ++a) w[a] = load(wealth, a);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const RowBuffer b = row_buffer(targets + (p < steps ? p : 0) * row, n);
#pragma unroll
    for (int a = 0; a < A; ++a) target[p][a] = load(b, a);
  }
  for (int32_t t0 = 0; t0 < steps; t0 += P) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int32_t t = t0 + p;
      if (t >= steps) break;
      uint32_t *inc = lds_inc + ((t & 1) ? words : 0);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const uint32_t to = target[p][a];
        if (w[a]) {
          if constexpr (kPacked)
            atomicAdd(&inc[to >> 1], 1u << ((to & 1u) << 4));
          else
            atomicAdd(&inc[to], 1u);
        }
      }
      // rows past the end: the last one again, not used
      const RowBuffer next = row_buffer(targets + (t + P < steps ? t + P : steps - 1) * row, n);
#pragma unroll
      for (int a = 0; a < A; ++a) target[p][a] = load(next, a);
      lds_barrier();  // what a step reads back goes through LDS
      const RowBuffer now = row_buffer(targets + t * row, n);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        uint32_t got;
        if constexpr (kPacked) {
          uint16_t *mine = reinterpret_cast<uint16_t *>(inc) + a * kWealthThreads + tid;
          got = *mine;
          *mine = 0;
        } else {
          uint32_t *mine = inc + a * kWealthThreads + tid;
          got = *mine;
          *mine = 0;
        }
        w[a] = w[a] - (w[a] < 1u ? w[a] : 1u) + got;
        store(now, a, w[a]);
      }
    }
  }
  const RowBuffer wealth = row_buffer(in.w, n);
#pragma unroll
  for (int a = 0; a < A; ++a) store(wealth, a, w[a]);
}

// Workgroups 0 .. count - 1 run the exchange chain of one instance each; the
// workgroups after them walk the positions of 1024 agents each, which only
// their own draws decide.  The chain is bound by its LDS latencies (atomic,
// barrier, read) up to about 2,000 agents and by the LDS accesses of one CU
// above.  1,000 agents x 100 steps: 25 us, where the workgroup that also
// walked, counted and ranked took 141; 5,003 x 150: 94 us and 1,768.
template <int A, bool kPacked>
__global__ void __launch_bounds__(kWealthThreads)
    k_wealth_exchange(const abm_wealth_inst *__restrict__ insts, int32_t count, int64_t cap) {
  extern __shared__ uint32_t lds_inc[];
  const int tid = threadIdx.x;
  if ((int32_t)blockIdx.x >= count) {
    const int32_t q = (int32_t)blockIdx.x - count;
    const abm_wealth_inst in = insts[q % count];
    const int64_t n = in.n, i = (int64_t)(q / count) * kWealthThreads + tid;
    if (!wealth_split_run(in, cap) || i >= n) return;
    constexpr int kAhead = 8;
    const GlobalPtr<uint32_t> draws = as_global(in.draws) + i;
    const GlobalPtr<float> gx = as_global(in.x) + i, gy = as_global(in.y) + i;
    float x = *gx, y = *gy;
    for (int32_t t0 = 0; t0 < in.steps; t0 += kAhead) {
      float dx[kAhead], dy[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int32_t t = t0 + k < in.steps ? t0 + k : in.steps - 1;
        dx[k] = __uint_as_float(draws[(int64_t)t * 3 * n]);
        dy[k] = __uint_as_float(draws[(int64_t)t * 3 * n + n]);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (t0 + k < in.steps) {
          x = mod1(x + dx[k]);
          y = mod1(y + dy[k]);
        }
    }
    *gx = x;
    *gy = y;
    return;
  }
  const abm_wealth_inst in = insts[blockIdx.x];
  // without steps there is no row of draws to load ahead
  if (!wealth_split_run(in, cap) || in.steps <= 0) return;
  for (int32_t k = tid; k < 2 * exchange_words(A, kPacked); k += kWealthThreads) lds_inc[k] = 0;
  __syncthreads();
  exchange_steps<A, kPacked>(in, lds_inc);
}

// ---- records of a run whose exchange is done
//
// Up to this many agents a wavefront takes a step's record alone, from a
// histogram of its own: a workgroup a record spends 10 us on barriers with most
// of its lanes idle, which a batch of small instances pays over and over (256
// instances of 1,000 agents x 100 steps: 542 us, and 162 for whole runs by a
// workgroup each).
constexpr int64_t kWaveRecordAgents = 1024;
constexpr int kWealthWaves = kWealthThreads / 64;
constexpr size_t kWaveRecordLds = kWealthWaves * (kWaveRecordAgents + 1) * 4;

// One wavefront records step t from the wealth row; hist: n + 1 bins in LDS,
// zero on entry and left zero.
__device__ __forceinline__ void wealth_wave_record(const abm_wealth_inst &in, int32_t t,
                                                   uint32_t *hist) {
  constexpr int kLoads = 8;  // in flight
  const int lane = threadIdx.x & 63;
  const int32_t n = (int32_t)in.n;
  const GlobalPtr<const uint32_t> row =
      as_global<const uint32_t>(in.draws) + (int64_t)t * 3 * n + 2 * n;
  for (int32_t i0 = lane; i0 - lane < n; i0 += 64 * kLoads) {
    uint32_t v[kLoads];
#pragma unroll
    for (int k = 0; k < kLoads; ++k) v[k] = row[min(i0 + 64 * k, n - 1)];
#pragma unroll
    for (int k = 0; k < kLoads; ++k)
      if (i0 + 64 * k < n) atomicAdd(&hist[v[k]], 1u);  // v <= n: wealth is conserved
  }
  // LDS operations of a wavefront complete in order; the compiler keeps it
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  uint32_t S = 0, T = 0, counted = 0;
  for (int32_t b = 0; counted < (uint32_t)n && b <= n; b += 64) {
    const int32_t w = b + lane;
    const uint32_t c = w <= n ? hist[w] : 0u;
    if (c) hist[w] = 0;
    uint32_t inc = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off);
      if (lane >= off) inc += y;
    }
    const uint32_t before = counted + inc - c;
    S += (uint32_t)w * (uint32_t)((uint64_t)c * before + (uint64_t)c * (c + 1) / 2);
    T += (uint32_t)w * c;
    counted += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    S += __shfl_xor(S, off);
    T += __shfl_xor(T, off);
  }
  if (lane == 0) wealth_write_record(in, t, T, S);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// LDS limit of the records: n + 1 bins, or the state of kWealthLdsAgents.
constexpr int64_t kRecordsLds = (kExchangeAgents + 1) * 4;
static_assert(kRecordsLds >= kWealthLdsAgents * kWealthLdsBytesPerAgent + 4 &&
                  kRecordsLds >= (int64_t)kWaveRecordLds && kRecordsLds + 128 <= 160 * 1024,
              "records LDS");

// Workgroup (b, instance): the records of steps b, b + gridDim.x, .. of an
// instance whose exchange has run, each from a histogram of the step's wealth
// row in LDS (n + 1 bins), a step a wavefront for few agents (the first
// wavefront of every workgroup first, then the second).  Workgroup 0 of an instance that the exchange
// kernel did not take runs it whole instead, in LDS where lds_bytes allow.
__global__ void __launch_bounds__(kWealthThreads)
    k_wealth_records(const abm_wealth_inst *__restrict__ insts, int64_t cap, int64_t lds_agents,
                     int mode) {
  extern __shared__ int32_t lds_agents_mem[];
  __shared__ uint32_t red[16];
  __shared__ uint32_t carry;
  const abm_wealth_inst in = insts[blockIdx.y];
  const int64_t n = in.n;
  const int tid = threadIdx.x;
  if (wealth_split_run(in, cap)) {
    int32_t *hist = lds_agents_mem;
    if ((int32_t)blockIdx.x >= in.steps) return;
    if (n <= kWaveRecordAgents) {
      const int32_t wave = tid >> 6;
      uint32_t *mine = reinterpret_cast<uint32_t *>(lds_agents_mem) + wave * (n + 1);
      for (int32_t b = tid & 63; b <= n; b += 64) mine[b] = 0;
      for (int32_t t = blockIdx.x + wave * gridDim.x; t < in.steps; t += kWealthWaves * gridDim.x)
        wealth_wave_record(in, t, mine);
      return;
    }
    for (int64_t b = tid; b <= n; b += kWealthThreads) hist[b] = 0;
    __syncthreads();
    for (int32_t t = blockIdx.x; t < in.steps; t += gridDim.x) {
      const GlobalPtr<const uint32_t> row =
          as_global<const uint32_t>(in.draws) + (int64_t)t * 3 * n + 2 * n;
      uint32_t total = 0;
      for (int64_t i = tid; i < n; i += kWealthThreads) {
        const uint32_t wi = row[i];
        atomicAdd(&hist[wi], 1);  // 0 <= wi <= n: wealth is conserved
        total += wi;
      }
      const uint32_t T = block_sum_u32(total, red);
      const uint32_t S = wealth_rank_sum(hist, n, red, carry);
      if (tid == 0) wealth_write_record(in, t, T, S);
      __syncthreads();
    }
    return;
  }
  if (blockIdx.x != 0) return;
  if (n <= lds_agents) {
    float *lx = reinterpret_cast<float *>(lds_agents_mem);
    float *ly = lx + n;
    int32_t *lw = reinterpret_cast<int32_t *>(ly + n);
    int32_t *linc = lw + n;
    int32_t *lhist = linc + n;
    for (int64_t i = tid; i < n; i += kWealthThreads) {
      lx[i] = in.x[i];
      ly[i] = in.y[i];
      lw[i] = in.w[i];
      linc[i] = 0;
      lhist[i] = 0;
    }
    if (tid == 0) lhist[n] = 0;
    __syncthreads();
    wealth_steps(in, lx, ly, lw, linc, lhist, red, carry, mode);
    for (int64_t i = tid; i < n; i += kWealthThreads) {
      in.x[i] = lx[i];
      in.y[i] = ly[i];
      in.w[i] = lw[i];
    }
  } else {
    wealth_steps(in, in.x, in.y, in.w, in.inc, in.hist, red, carry, mode);
  }
}

// ---- one large instance across the whole GPU (abm_wealth_run_grid): one launch
// per step with scratch for second copies (k_wealth_grid_step, below), two
// without.  K1(t): every workgroup draws step t for its agents and applies the
// draws (positions; one exchange atomic per giving agent), and workgroup 0 first
// records step t-1 from the histogram.  K2(t): the exchange is applied and the
// wealth histogram built.  Either way wealth stays bunched on a few small values,
// so the histogram is gathered without hot words: per-workgroup LDS bins, flushed
// with one atomic per bin in use, the values below kGridHot into one of
// kGridCopies copies (chosen by workgroup) and the rest into the instance's
// histogram.  The total T is conserved, so it is summed once, at step 0; the
// record stops once it has counted all n agents, so no running maximum is kept.
// The same integer and IEEE float operations as the one-workgroup run, so the
// same bits.
constexpr int kGridThreads = 256;
constexpr int kGridBins = 1024;     // LDS histogram bins per workgroup
constexpr int64_t kGridMaxBlocks = 1024;
// workgroups of a one-launch step, beside the recording one (each flushes its
// bins, so a large instance gives them several tiles of agents)
constexpr int64_t kGridStepBlocks = 4096;
// a one-launch step's scratch, 2 n + 1 + 1024 + 8 words, is within 3 n from here
constexpr int64_t kGridOneLaunch = 1033;
constexpr int kGridHot = 64;        // values with their own histogram copies
constexpr int kGridCopies = 16;
static_assert(ABM_WEALTH_GRID_ACC_WORDS == 2 + kGridCopies * kGridHot,
              "acc layout: T, a spare word, then the hot-bin copies");

// Mean and Gini of step t from a histogram set and the total; clears the bins it
// reads (one workgroup).  Bins are read 256 a round until all n agents are
// counted, which covers every nonzero bin.
__device__ void wealth_grid_rank(const abm_wealth_inst &in, int32_t t, uint32_t T, uint32_t *hot,
                                 uint32_t *hist, uint32_t *red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n = in.n;
  uint32_t S_part = 0, counted = 0;
  for (int64_t base = 0; base <= n; base += kGridThreads) {
    const int64_t w = base + tid;
    uint32_t c = 0;
    if (w < kGridHot) {
      uint32_t v[kGridCopies];
#pragma unroll
      for (int k = 0; k < kGridCopies; ++k) v[k] = hot[k * kGridHot + w];
#pragma unroll
      for (int k = 0; k < kGridCopies; ++k) {
        c += v[k];
        if (v[k]) hot[k * kGridHot + w] = 0;
      }
    } else if (w <= n) {
      c = hist[w];
      if (c) hist[w] = 0;
    }
    uint32_t inc = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off);
      if (lane >= off) inc += y;
    }
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    uint32_t before = counted + inc - c;
    for (int q = 0; q < kGridThreads / 64; ++q) {
      if (q < wave) before += red[q];
      counted += red[q];
    }
    if (c) {
      const uint64_t ranksum = (uint64_t)c * before + (uint64_t)c * (c + 1) / 2;
      S_part += (uint32_t)w * (uint32_t)ranksum;
    }
    __syncthreads();  // red is rewritten
    if ((int64_t)counted >= n) break;  // block-uniform
  }
  const uint32_t S = block_sum_u32(S_part, red);
  if (tid == 0) wealth_write_record(in, t, T, S);
}

__global__ void __launch_bounds__(kGridThreads)
    k_wealth_grid_agents(abm_wealth_inst in, int32_t t, uint32_t *acc, int mode) {
  __shared__ uint32_t red[kGridThreads / 64];
  if (blockIdx.x == 0 && t > 0)
    wealth_grid_rank(in, t - 1, acc[0], acc + 2, (uint32_t *)in.hist, red);
  if (t >= in.steps) return;
  const int64_t n = in.n;
  const int64_t stride = (int64_t)gridDim.x * kGridThreads;
  for (int64_t i = (int64_t)blockIdx.x * kGridThreads + threadIdx.x; i < n; i += stride) {
    // the unit first: see k_wealth_grid_step
    Key kk1, kk2;
    target_keys(in.keys, t, kk1, kk2, mode);
    const uint32_t target = wealth_target(kk1, kk2, n, i, mode);
    if (in.w[i] > 0) atomicAdd(&in.inc[target], 1);
    const WealthWalk d = wealth_walk(collection_key(in.keys, t), n, i, mode);
    in.x[i] = mod1(in.x[i] + d.mdx);
    in.y[i] = mod1(in.y[i] + d.mdy);
  }
}

__global__ void __launch_bounds__(kGridThreads)
    k_wealth_grid_apply(abm_wealth_inst in, uint32_t *acc, int32_t t) {
  __shared__ uint32_t red[kGridThreads / 64];
  __shared__ uint32_t bins[kGridBins];
  for (int b = threadIdx.x; b < kGridBins; b += kGridThreads) bins[b] = 0;
  __syncthreads();
  const int64_t n = in.n;
  const int64_t stride = (int64_t)gridDim.x * kGridThreads;
  uint32_t total = 0;
  for (int64_t i = (int64_t)blockIdx.x * kGridThreads + threadIdx.x; i < n; i += stride) {
    const int32_t w0 = in.w[i];
    const int32_t wi = w0 - (w0 > 0 ? 1 : 0) + in.inc[i];
    in.w[i] = wi;
    in.inc[i] = 0;
    // 0 <= wi <= n: wealth is conserved
    if (wi < kGridBins)
      atomicAdd(&bins[wi], 1u);
    else
      atomicAdd(&in.hist[wi], 1);
    total += (uint32_t)wi;
  }
  __syncthreads();
  uint32_t *hot = acc + 2 + (int64_t)(blockIdx.x % kGridCopies) * kGridHot;
  for (int b = threadIdx.x; b < kGridBins; b += kGridThreads) {
    const uint32_t c = bins[b];
    if (!c) continue;
    if (b < kGridHot)
      atomicAdd(&hot[b], c);
    else
      atomicAdd(&in.hist[b], (int32_t)c);
  }
  if (t == 0) {  // the total, conserved from here on
    const uint32_t T = block_sum_u32(total, red);
    if (threadIdx.x == 0) atomicAdd(&acc[0], T);
  }
}

// One launch per step, with scratch for a second increment array, histogram
// and set of hot bins: launch t applies step t - 1's exchange to its agents
// (own reads and writes only) and counts their wealth, then gives step t's
// units and walks, and workgroup 0 records step t - 2.  What a launch adds to
// (increments of step t, bins of step t - 1) and what it reads and clears
// (increments of step t - 1, bins of step t - 2) alternate between the two
// copies, so no launch reads what another workgroup of it writes.  Launch
// `steps` only applies, launch steps + 1 only records.  A step of 247,720
// agents takes 11.0 us: 5.0 without the walk and the exchange's atomics, of
// which the 156,000 (26 per ns, whatever their scope) take 5.9 and the walk's
// five threefry blocks and two erf_inv 4.8 beside them.  Two launches a step,
// with the record in front of workgroup 0's agents, took 14.0.
// The keys that all agents share (split(uk) of the step) are made by workgroup
// 0 of the launch before; in every thread they were 137 of 990 operations.
struct WealthGrid {
  uint32_t *inc[2], *hist[2], *hot[2], *total;
  uint32_t *shared_keys;  // [2][4]: kk1, kk2 of even and odd steps
};

// split(uk) of step t into the shared keys (one thread).
__device__ __forceinline__ void wealth_shared_keys(const abm_wealth_inst &in, uint32_t *shared,
                                                   int32_t t, int mode) {
  Key kk1, kk2;
  split2(Key{in.keys[4 * t + 2], in.keys[4 * t + 3]}, kk1, kk2, mode);
  uint32_t *out = shared + 4 * (t & 1);
  out[0] = kk1.k0;
  out[1] = kk1.k1;
  out[2] = kk2.k0;
  out[3] = kk2.k1;
}

template <int kMode>
__global__ void __launch_bounds__(kGridThreads)
    k_wealth_grid_step(abm_wealth_inst in, WealthGrid g, int32_t t) {
  __shared__ uint32_t red[kGridThreads / 64];
  __shared__ uint32_t bins[kGridBins];
  const int64_t n = in.n;
  const int cur = t & 1, prev = cur ^ 1;
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0 && t + 1 < in.steps)
      wealth_shared_keys(in, g.shared_keys, t + 1, kMode);
    if (t > 1) wealth_grid_rank(in, t - 2, *g.total, g.hot[cur], g.hist[cur], red);
    return;
  }
  if (t > in.steps) return;
  for (int b = threadIdx.x; b < kGridBins; b += kGridThreads) bins[b] = 0;
  __syncthreads();
  uint32_t total = 0;
  const int32_t tk = t < in.steps ? t : 0;  // the last launch draws nothing
  const Key ck{in.keys[4 * tk], in.keys[4 * tk + 1]};
  const uint32_t *sk = g.shared_keys + 4 * (tk & 1);
  const Key kk1{sk[0], sk[1]}, kk2{sk[2], sk[3]};
  const int64_t stride = (int64_t)(gridDim.x - 1) * kGridThreads;
#pragma unroll 1
  for (int64_t i = (int64_t)(blockIdx.x - 1) * kGridThreads + threadIdx.x; i < n; i += stride) {
    int32_t wi = in.w[i];
    if (t > 0) {
      wi = wi - (wi > 0 ? 1 : 0) + (int32_t)g.inc[prev][i];
      g.inc[prev][i] = 0;
      in.w[i] = wi;
      // 0 <= wi <= n: wealth is conserved
      if (wi < kGridBins)
        atomicAdd(&bins[wi], 1u);
      else
        atomicAdd(&g.hist[prev][wi], 1u);
      total += (uint32_t)wi;
    }
    if (t < in.steps) {
      // the unit first, so that its atomic runs beside the walk's draws
      const uint32_t target = wealth_target(kk1, kk2, n, i, kMode);
      if (wi > 0) atomicAdd(&g.inc[cur][target], 1u);
      const WealthWalk d = wealth_walk(ck, n, i, kMode);
      in.x[i] = mod1(in.x[i] + d.mdx);
      in.y[i] = mod1(in.y[i] + d.mdy);
    }
  }
  if (t == 0) return;
  __syncthreads();
  uint32_t *hot = g.hot[prev] + (int64_t)(blockIdx.x % kGridCopies) * kGridHot;
  for (int b = threadIdx.x; b < kGridBins; b += kGridThreads) {
    const uint32_t c = bins[b];
    if (!c) continue;
    atomicAdd(b < kGridHot ? &hot[b] : &g.hist[prev][b], c);
  }
  if (t == 1) {  // the total, conserved from here on
    const uint32_t T = block_sum_u32(total, red);
    if (threadIdx.x == 0) atomicAdd(g.total, T);
  }
}

// Clears a run's scratch and makes step 0's shared keys.
__global__ void k_wealth_grid_begin(abm_wealth_inst in, WealthGrid g, uint32_t *acc, int64_t used,
                                    int mode) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < used) in.draws[i] = 0;
  if (i < ABM_WEALTH_GRID_ACC_WORDS) acc[i] = 0;
  if (i == used) wealth_shared_keys(in, g.shared_keys, 0, mode);
}

__global__ void k_wealth_zero_acc(uint32_t *acc) {
  for (int i = threadIdx.x; i < ABM_WEALTH_GRID_ACC_WORDS; i += blockDim.x) acc[i] = 0;
}

__global__ void k_wealth_init(const uint32_t *__restrict__ init_key, Key key, int64_t n,
                              float *__restrict__ x, float *__restrict__ y,
                              int32_t *__restrict__ w, int mode) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (init_key) key = Key{init_key[0], init_key[1]};
  Key kx, ky;
  split2(split_at(key, n, i, mode), kx, ky, mode);
  x[i] = unit_float(bits_scalar(kx, mode));
  y[i] = unit_float(bits_scalar(ky, mode));
  w[i] = 1;
}

using ExchangeKernel = void (*)(const abm_wealth_inst *, int32_t, int64_t);

// One instantiation per number of agents a thread keeps.
struct ExchangeVariant {
  int agents;
  size_t lds;
  ExchangeKernel kernel;
};
template <int A, bool kPacked>
constexpr ExchangeVariant exchange_variant() {
  return ExchangeVariant{A, 8 * (size_t)exchange_words(A, kPacked), k_wealth_exchange<A, kPacked>};
}
const ExchangeVariant kExchange[] = {
    exchange_variant<1, false>(),  exchange_variant<2, false>(),  exchange_variant<3, false>(),
    exchange_variant<4, false>(),  exchange_variant<5, false>(),  exchange_variant<6, false>(),
    exchange_variant<8, false>(),  exchange_variant<10, false>(), exchange_variant<12, false>(),
    exchange_variant<16, false>(), exchange_variant<20, false>(), exchange_variant<24, true>(),
    exchange_variant<32, true>(),  exchange_variant<40, true>()};

// Instances of a launch that has a grid row for each.
constexpr int32_t kGridRows = 65535;

// Workgroups of the draws kernel for each of `count` instances.  A draw is a
// chain of about 900 dependent operations, so a SIMD wants its 8 wavefronts:
// 2,048 workgroups fill the chip (5,003 x 150: 29 us, 33 with 512); many
// instances fill it with 512 each.
unsigned draw_blocks(int32_t count) {
  return (unsigned)std::max(512, std::min(2048, 4096 / std::max(count, 1)));
}

// Workgroups of the records for each of `count` instances: a lone one has its
// steps on as many CUs, many share a few thousand workgroups (256 for each of
// 4,096 cost 2.5 ms to launch, most of them without a step).
unsigned record_blocks(int32_t count) {
  return (unsigned)std::max(1, std::min(256, 4096 / count));
}

// These kernels may need more than 64 KB of dynamic LDS: the limits are
// raised once per device, under a lock.
constexpr int kMaxDevices = 64;
std::mutex g_wealth_attr_mu;
bool g_wealth_attr_set[kMaxDevices];

int wealth_lds_attr() {
  int dev = -1;
  ABM_CHECK_HIP(hipGetDevice(&dev));
  ABM_REQUIRE(dev >= 0 && dev < kMaxDevices, "wealth: device index out of range");
  std::lock_guard<std::mutex> lock(g_wealth_attr_mu);
  if (!g_wealth_attr_set[dev]) {
    for (const ExchangeVariant &v : kExchange)
      ABM_CHECK_HIP(hipFuncSetAttribute((const void *)v.kernel,
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)v.lds));
    ABM_CHECK_HIP(hipFuncSetAttribute((const void *)k_wealth_records,
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)kRecordsLds));
    g_wealth_attr_set[dev] = true;
  }
  return kOk;
}

}  // namespace abm

using namespace abm;

extern "C" {

int abm_wealth_init(const uint32_t *init_key, int64_t n, float *x, float *y, int32_t *w,
                    int mode, void *stream) {
  ABM_REQUIRE(init_key && x && y && w && n > 1 && n < (1ll << 31) &&
                  (mode == 0 || mode == 1),
              "abm_wealth_init: bad arguments");
  hipLaunchKernelGGL(k_wealth_init, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, init_key, Key{0u, 0u}, n, x, y, w, mode);
  ABM_LAUNCH_CHECK("abm_wealth_init");
  return kOk;
}

int abm_wealth_init_host_key(const uint32_t init_key[2], int64_t n, float *x, float *y, int32_t *w,
                             int mode, void *stream) {
  ABM_REQUIRE(init_key && x && y && w && n > 1 && n < (1ll << 31) &&
                  (mode == 0 || mode == 1),
              "abm_wealth_init_host_key: bad arguments");
  hipLaunchKernelGGL(k_wealth_init, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const uint32_t *)nullptr, Key{init_key[0], init_key[1]},
                     n, x, y, w, mode);
  ABM_LAUNCH_CHECK("abm_wealth_init_host_key");
  return kOk;
}

int abm_wealth_run_grid(const abm_wealth_inst *inst, uint32_t *acc, int mode, void *stream) {
  ABM_REQUIRE(inst && acc && (mode == 0 || mode == 1), "abm_wealth_run_grid: bad arguments");
  const abm_wealth_inst in = *inst;
  ABM_REQUIRE(in.n >= 2 && in.n < (1ll << 31) && in.steps >= 0 && in.x && in.y && in.w &&
                  in.inc && in.hist && in.keys && in.mean_out && in.gini_out,
              "abm_wealth_run_grid: incomplete instance");
  hipStream_t s = (hipStream_t)stream;
  if (in.steps == 0) return kOk;
  if (in.draws && in.n >= kGridOneLaunch) {
    WealthGrid g;
    g.total = acc;
    g.inc[0] = (uint32_t *)in.inc;
    g.hist[0] = (uint32_t *)in.hist;
    g.hot[0] = acc + 2;
    g.inc[1] = in.draws;
    g.hist[1] = in.draws + in.n;
    g.hot[1] = in.draws + 2 * in.n + 1;
    const int64_t used = 2 * in.n + 1 + kGridCopies * kGridHot;
    g.shared_keys = in.draws + used;
    hipLaunchKernelGGL(k_wealth_grid_begin, dim3((unsigned)(used / 256 + 1)), dim3(256), 0, s, in,
                       g, acc, used, mode);
    const int64_t tiles = (in.n + kGridThreads - 1) / kGridThreads;
    const int64_t per = (tiles + kGridStepBlocks - 1) / kGridStepBlocks;  // tiles a workgroup
    const unsigned blocks = (unsigned)(1 + (tiles + per - 1) / per);
    auto *step = mode == kModePartitionable ? k_wealth_grid_step<kModePartitionable>
                                            : k_wealth_grid_step<kModeOriginal>;
    for (int32_t t = 0; t <= in.steps + 1; ++t)  // the last one only records
      hipLaunchKernelGGL(step, dim3(t <= in.steps ? blocks : 1), dim3(kGridThreads), 0, s, in, g,
                         t);
    ABM_LAUNCH_CHECK("abm_wealth_run_grid");
    return kOk;
  }
  hipLaunchKernelGGL(k_wealth_zero_acc, dim3(1), dim3(256), 0, s, acc);
  int64_t blocks = (in.n + kGridThreads - 1) / kGridThreads;
  if (blocks > kGridMaxBlocks) blocks = kGridMaxBlocks;
  for (int32_t t = 0; t <= in.steps; ++t) {
    hipLaunchKernelGGL(k_wealth_grid_agents, dim3((unsigned)blocks), dim3(kGridThreads), 0, s,
                       in, t, acc, mode);
    if (t < in.steps)
      hipLaunchKernelGGL(k_wealth_grid_apply, dim3((unsigned)blocks), dim3(kGridThreads), 0, s,
                         in, acc, t);
  }
  ABM_LAUNCH_CHECK("abm_wealth_run_grid");
  return kOk;
}

int abm_wealth_run_batch(const abm_wealth_inst *insts, int32_t count, int64_t max_n, int mode,
                         void *stream) {
  ABM_REQUIRE(insts && count >= 0 && max_n >= 0 && (mode == 0 || mode == 1),
              "abm_wealth_run_batch: bad arguments");
  if (count == 0) return kOk;
  if (int rc = wealth_lds_attr()) return rc;
  hipStream_t s = (hipStream_t)stream;
  // the exchange kernel takes instances of up to `cap` agents: the table's
  // largest, and always those of one agent per thread
  const int64_t known = max_n <= kExchangeAgents ? max_n : 0;
  const int64_t cap = known > kWealthThreads ? known : kWealthThreads;
  const int per = (int)((cap + kWealthThreads - 1) / kWealthThreads);
  const ExchangeVariant *v = kExchange;
  while (v->agents < per) ++v;
  // LDS of the records: the histogram of `cap` agents, or the whole state of
  // an instance that runs in one workgroup (no draw buffer)
  const int64_t lds_agents = max_n > 0 && max_n <= kWealthLdsAgents ? max_n : 0;
  size_t dyn = (size_t)(lds_agents * kWealthLdsBytesPerAgent + 4);
  if (dyn < (size_t)(cap + 1) * 4) dyn = (size_t)(cap + 1) * 4;
  if (dyn < kWaveRecordLds) dyn = kWaveRecordLds;
  for (int32_t done = 0; done < count; done += kGridRows) {
    const abm_wealth_inst *part = insts + done;
    const int32_t rows = std::min(count - done, kGridRows);
    hipLaunchKernelGGL(mode == kModePartitionable ? k_wealth_draws<kModePartitionable>
                                                  : k_wealth_draws<kModeOriginal>,
                       dim3(draw_blocks(rows), (unsigned)rows), dim3(kDrawThreads), 0, s, part);
    hipLaunchKernelGGL(v->kernel, dim3((unsigned)(rows * (1 + per))), dim3(kWealthThreads),
                       v->lds, s, part, rows, cap);
    hipLaunchKernelGGL(k_wealth_records, dim3(record_blocks(rows), (unsigned)rows),
                       dim3(kWealthThreads), dyn, s, part, cap, lds_agents, mode);
  }
  ABM_LAUNCH_CHECK("abm_wealth_run_batch");
  return kOk;
}

}  // extern "C"
