// schelling.hip -- Schelling segregation on a periodic Grid.
//
// Program (reference Grid stores only shape and the periodic flag,
// jaxabm/agentpy.py:465-527; step schedule jaxabm/model.py:146-216):
//  init   u = uniform(PRNGKey(seed), (H*W,)); cell type 1 if u < 0.45, 2 if
//         u < 0.9, else empty; agent k = k-th occupied cell in row-major order
//  step   empty list = empty cells of the pre-step grid in row-major order;
//         agent phase (agent keys = split(ck, n_agents)): Moore-8 on the torus,
//         happy iff 8 * same >= 3 * occupied (same/occupied >= 0.375, an
//         isolated agent is happy); an unhappy agent draws
//         j = randint(agent_key, (), 0, n_empty) and claims empty[j];
//         env phase: each claimed cell goes to its lowest-id claimant, winners
//         move (their old cell is not reusable until the next step)
//  record fraction happy (agent phase) and number of moves
//
// The empty cells are kept as a bitmap (bit c set when cell c is empty) and a
// count per 1024-cell block; the moves kernel keeps both current with atomics
// (a bit flip per moved agent, and a count update when a move crosses blocks;
// a cell changes state at most once per step), so the row-major empty list is
// never materialised: every agents block scans the block counts (1 KB at
// 512 x 512) into an LDS prefix, and empty[j] is then a search of that prefix
// and a popcount scan of one block's 32 bitmap words.  Two kernels per step
// (captured with the rest of the run; small grids run in one launch, below):
//   k_schelling_agents  32x32 cell tiles + 1-cell torus halo in LDS;
//                       happiness, draw, empty[j], atomicMin claim
//   k_schelling_moves   winners move; bitmap, block counts and claims updated
// Layout (HBM): cells int8[H*W], id int32[H*W] (agent on a cell or -1),
// claim int32[H*W] (INT32_MAX when unclaimed), pos int32[n_agents],
// type int8[n_agents], target int32[n_agents], empty-cell bitmap
// uint32[32 * ceil(H*W/1024)] (in the grid's `empty` scratch), empty cells per
// 1024-cell block int32[16][ceil(H*W/1024)] (16 copies summed by readers; in
// the `block_counts` scratch).
#include <hip/hip_runtime.h>

#include <climits>
#include <mutex>

#define ABM_STRAIGHT_DRAWS
#include "common.hpp"
#include "jaxabm_amd.h"
#include "watch.hpp"

namespace abm {

constexpr int kTileDim = 32;
constexpr int kCellsPerBlock = 1024;
constexpr int kWordsPerBlock = kCellsPerBlock / 32;
// block prefix of the empty counts in LDS: with the agents kernel's 5.3 KB of
// static LDS, at most 64 KB in all
constexpr int64_t kMaxEmptyBlocks = 15000;
// copies of the per-block empty counts: the moves kernel's workgroup w updates
// copy w % kCountCopies, so the count atomics of a busy step spread over 16x
// the words (each word's device-scope atomics serialise); readers sum them
constexpr int kCountCopies = 16;

// number of cells with (cells[c] == 0) == want_empty per 1024-cell block
__global__ void __launch_bounds__(kCellsPerBlock)
    k_cells_count(const int8_t *__restrict__ cells, int64_t nc, int want_empty,
                  int32_t *__restrict__ block_counts) {
  const int64_t c = (int64_t)blockIdx.x * kCellsPerBlock + threadIdx.x;
  const bool hit = c < nc && ((cells[c] == 0) == (want_empty != 0));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __shared__ int32_t wc[16];
  const uint64_t m = __ballot(hit);
  if (lane == 0) wc[wave] = (int32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t s = 0;
    for (int w = 0; w < 16; ++w) s += wc[w];
    block_counts[blockIdx.x] = s;
  }
}

// Writes the matching cells in row-major order: out[rank] = cell.  When
// agent arrays are given (init), also numbers the agents: pos, type, id.
__global__ void __launch_bounds__(kCellsPerBlock)
    k_cells_scatter(const int8_t *__restrict__ cells, int64_t nc, int want_empty,
                    const int32_t *__restrict__ block_counts, int32_t *__restrict__ out,
                    int8_t *__restrict__ type, int32_t *__restrict__ id) {
  __shared__ int32_t base;
  __shared__ int32_t wc[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // block offset = sum of the counts of earlier blocks
  int32_t part = 0;
  for (int32_t b = tid; b < (int32_t)blockIdx.x; b += kCellsPerBlock) part += block_counts[b];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off);
  if (lane == 0) wc[wave] = part;
  __syncthreads();
  if (tid == 0) {
    int32_t s = 0;
    for (int w = 0; w < 16; ++w) s += wc[w];
    base = s;
  }
  __syncthreads();
  const int64_t c = (int64_t)blockIdx.x * kCellsPerBlock + tid;
  const bool hit = c < nc && ((cells[c] == 0) == (want_empty != 0));
  const uint64_t m = __ballot(hit);
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  __syncthreads();
  if (lane == 0) wc[wave] = (int32_t)__popcll(m);
  __syncthreads();
  int32_t before = base;
  for (int w = 0; w < wave; ++w) before += wc[w];
  if (hit) {
    const int32_t r = before + (int32_t)__popcll(m & lt);
    out[r] = (int32_t)c;
    if (type) type[r] = cells[c];
    if (id) id[c] = r;
  } else if (id && c < nc) {
    id[c] = -1;
  }
}

// Empty-cell bitmap of the current grid: one ballot per 64 cells; cells past
// the last one are not empty.
__global__ void __launch_bounds__(kCellsPerBlock)
    k_empty_bits(const int8_t *__restrict__ cells, int64_t nc, uint32_t *__restrict__ ebits) {
  const int64_t c = (int64_t)blockIdx.x * kCellsPerBlock + threadIdx.x;
  const bool e = c < nc && cells[c] == 0;
  const uint64_t m = __ballot(e);
  if ((threadIdx.x & 63) == 0) {
    const int64_t w = c >> 5;  // c is the wave's first cell (a multiple of 64)
    ebits[w] = (uint32_t)m;
    ebits[w + 1] = (uint32_t)(m >> 32);
  }
}

// Empty cells of block b < nb: the sum of its count copies.
__device__ __forceinline__ int32_t block_empty(const int32_t *__restrict__ ecount, int nb,
                                               int b) {
  int32_t v[kCountCopies];
#pragma unroll
  for (int r = 0; r < kCountCopies; ++r) v[r] = ecount[(int64_t)r * nb + b];
  int32_t s = 0;
#pragma unroll
  for (int r = 0; r < kCountCopies; ++r) s += v[r];
  return s;
}

// P[0] = 0, P[b + 1] = empty cells of blocks 0 .. b, for b < nb, in LDS, from
// the per-block counts (wave scans).  first: this thread's count for the
// first chunk of blockDim.x blocks, loaded by the caller ahead of its other
// loads.  Up to blockDim.x blocks (grids of up to 1M cells at 1024 threads)
// the scan takes two barriers; larger grids scan chunk by chunk.
__device__ void empty_prefix(const int32_t *__restrict__ ecount, int nb, int32_t first,
                             int32_t *P, int32_t *wsum, int32_t *carry) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nthreads = (int)blockDim.x;
  if (nb <= nthreads) {
    int32_t v = first;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(v, off);
      if (lane >= off) v += y;
    }
    if (lane == 63) wsum[wave] = v;
    if (tid == 0) P[0] = 0;
    __syncthreads();
    if (tid < nb) {
      int32_t before = 0;
      for (int q = 0; q < wave; ++q) before += wsum[q];
      P[tid + 1] = before + v;
    }
    __syncthreads();
    return;
  }
  if (tid == 0) {
    P[0] = 0;
    *carry = 0;
  }
  __syncthreads();
  for (int base = 0; base < nb; base += nthreads) {
    const int b = base + tid;
    int32_t v = base == 0 ? first : (b < nb ? block_empty(ecount, nb, b) : 0);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(v, off);
      if (lane >= off) v += y;
    }
    if (lane == 63) wsum[wave] = v;
    __syncthreads();
    int32_t before = *carry;
    for (int q = 0; q < wave; ++q) before += wsum[q];
    if (b < nb) P[b + 1] = before + v;
    __syncthreads();
    if (tid == nthreads - 1) *carry = before + v;
    __syncthreads();
  }
}

// Cell of the j-th empty cell in row-major order (j < P[nb]): the block b with
// P[b] <= j < P[b + 1], then the (j - P[b])-th set bit of its 32 bitmap words,
// one cache line, read 16 bytes at a time.
__device__ __forceinline__ int32_t jth_empty(uint32_t j, const int32_t *P, int nb,
                                             const uint32_t *__restrict__ ebits) {
  int lo = 0, hi = nb;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((uint32_t)P[mid] <= j)
      lo = mid;
    else
      hi = mid;
  }
  uint32_t r = j - (uint32_t)P[lo];
  const int64_t w0 = (int64_t)lo * kWordsPerBlock;
  uint4 v[kWordsPerBlock / 4];
#pragma unroll
  for (int q = 0; q < kWordsPerBlock / 4; ++q) v[q] = reinterpret_cast<const uint4 *>(ebits + w0)[q];
  // the four words, then the word: the last with at most r bits before it
  uint32_t n = 0, before = 0, w = 0;
  uint4 four = v[0];
#pragma unroll
  for (int q = 0; q < kWordsPerBlock / 4; ++q) {
    const bool here = n <= r;
    before = here ? n : before;
    four.x = here ? v[q].x : four.x;
    four.y = here ? v[q].y : four.y;
    four.z = here ? v[q].z : four.z;
    four.w = here ? v[q].w : four.w;
    w = here ? 4 * q : w;
    n += (uint32_t)(__popc(v[q].x) + __popc(v[q].y) + __popc(v[q].z) + __popc(v[q].w));
  }
  if (r >= n) return -1;
  const uint32_t words[4] = {four.x, four.y, four.z, four.w};
  uint32_t word = four.x;
  n = before;
  const uint32_t w4 = w;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool here = n <= r;
    before = here ? n : before;
    word = here ? words[q] : word;
    w = here ? w4 + q : w;
    n += (uint32_t)__popc(words[q]);
  }
  // the bit, by halves
  r -= before;
  uint32_t bit = 0;
#pragma unroll
  for (int half = 16; half > 0; half >>= 1) {
    const uint32_t low = (uint32_t)__popc((word >> bit) & ((1u << half) - 1));
    if (r >= low) {
      r -= low;
      bit += half;
    }
  }
  return (int32_t)((w0 + w) * 32 + bit);
}

struct SchellingStep {
  int32_t H, W;
  int64_t n_agents, n_empty;
  const int8_t *cells;
  const int32_t *id;
  const uint32_t *ebits;
  const int32_t *ecount;
  int32_t nb;
  int32_t *claim, *target;
  const uint32_t *ck;
  int32_t *happy_count;
  // the previous step's happy count (null at a run's first step): when every
  // agent was happy then, nobody moved, the grid is unchanged and this step
  // is the identity
  const int32_t *prev_happy;
  int32_t *watch;  // host words of a watched run, or null
  int32_t begun;   // value for watch[0], or 0: this step does not tell
};

// True when the step is the identity: the previous step found every agent
// happy, so nothing moved since and every agent is happy again.
__device__ __forceinline__ bool schelling_identity(const int32_t *prev_happy, int64_t n_agents) {
  return prev_happy && (int64_t)*prev_happy == n_agents;
}

// Bound by its chain, not by bytes or instructions: the step before's count, one
// round of loads, the prefix's barriers, the draw, the bitmap line, the claim's
// atomic, each from memory that another XCD wrote a launch before.  Two
// workgroups a CU (8 wavefronts a SIMD, 64 registers) pay from about 300,000
// cells on, but not with registers spilled: 40 steps of 1,030 x 1,030 took 1,331
// us before the loads left their branches, 1,122 now, 1,278 at 72 registers and
// 1,689 spilling; 200 steps of 512 x 512, all launched, 1,335 and 1,190.  (Bit
// planes of the whole grid read and scanned by every workgroup in place of
// counts, tiles and the search in memory took 779 us against 600 for 40 steps of
// 614 x 640.)
template <int kMode>
__global__ void __launch_bounds__(kTileDim * kTileDim, 8) k_schelling_agents(SchellingStep a) {
  extern __shared__ int32_t empty_prefix_lds[];  // [nb + 1]
  __shared__ int8_t tile[kTileDim + 2][kTileDim + 2];
  __shared__ int32_t wc[16];
  __shared__ int32_t carry;
  __shared__ int32_t work[kTileDim * kTileDim];  // the tile's agents that draw a target
  __shared__ int32_t nwork;
  constexpr int kHalo = (kTileDim + 2) * (kTileDim + 2);  // 34 x 34 cells, <= 2 per thread
  const int tid = threadIdx.x;
  const int tx = tid % kTileDim, ty = tid / kTileDim;
  const int r0 = blockIdx.y * kTileDim, c0 = blockIdx.x * kTileDim;
  const int r = r0 + ty, c = c0 + tx;
  const bool inside = r < a.H && c < a.W;
  const int64_t cell = (int64_t)r * a.W + c;
  // One memory round trip after the step before's count: the tile and its torus
  // halo, this thread's block counts for the prefix, the agent on its cell.  No
  // load is in a branch (one there waits for all before it): a thread without
  // a place of its own loads another's.
  const int32_t prev = *(a.prev_happy ? a.prev_happy : a.happy_count);
  int8_t tv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = min(tid + i * kTileDim * kTileDim, kHalo - 1);
    const int lr = q / (kTileDim + 2), lc = q % (kTileDim + 2);
    // r0 < H and c0 < W: at most 32 cells past the edge
    int gr = r0 + lr - 1 + a.H, gc = c0 + lc - 1 + a.W;
    if (a.H <= kTileDim) gr %= a.H;
    if (a.W <= kTileDim) gc %= a.W;
    gr -= gr >= a.H ? a.H : 0;
    gr -= gr >= a.H ? a.H : 0;
    gc -= gc >= a.W ? a.W : 0;
    gc -= gc >= a.W ? a.W : 0;
    tv[i] = a.cells[(int64_t)gr * a.W + gc];
  }
  const int block = min(tid, a.nb - 1);
  int32_t copies[kCountCopies];
#pragma unroll
  for (int q = 0; q < kCountCopies; ++q) copies[q] = a.ecount[(int64_t)q * a.nb + block];
  const int32_t id = a.id[inside ? cell : 0];
  if (a.prev_happy && prev == (int32_t)a.n_agents) {  // grid-uniform: the identity
    // every agent happy again; no target is drawn (the last step left each
    // agent's target at -1) and the moves kernel exits too
    if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) {
      *a.happy_count = (int32_t)a.n_agents;
      if (a.watch) tell_host(&a.watch[1], 1);  // which ends the host's wait too
    }
    return;
  }
  if (a.begun && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) tell_host(&a.watch[0], a.begun);
  const int32_t k = inside ? id : -1;
  int32_t first = 0;
  if (tid < a.nb) {
#pragma unroll
    for (int q = 0; q < kCountCopies; ++q) first += copies[q];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = tid + i * (int)blockDim.x;
    if (q < kHalo) tile[q / (kTileDim + 2)][q % (kTileDim + 2)] = tv[i];
  }
  if (tid == 0) nwork = 0;  // visible after the prefix's barriers
  empty_prefix(a.ecount, a.nb, first, empty_prefix_lds, wc, &carry);
  bool happy = false, draws = false;
  if (inside) {
    const int8_t me = tile[ty + 1][tx + 1];
    if (me) {
      int occ = 0, same = 0;
#pragma unroll
      for (int dr = -1; dr <= 1; ++dr)
#pragma unroll
        for (int dc = -1; dc <= 1; ++dc) {
          if (!dr && !dc) continue;
          const int8_t v = tile[ty + 1 + dr][tx + 1 + dc];
          occ += v != 0;
          same += v == me;
        }
      happy = 8 * same >= 3 * occ;
      draws = !happy && a.n_empty > 0;
      if (!draws) a.target[k] = -1;
    }
  }
  // The agents that draw go to the front of the workgroup, so that the draw
  // and the search run on full waves, not on every wave that holds one.
  const int lane = tid & 63;
  const uint64_t dm = __ballot(draws);
  if (dm) {  // wave-uniform
    int32_t base = 0;
    if (lane == 0) base = atomicAdd(&nwork, (int32_t)__popcll(dm));
    base = __shfl(base, 0);
    if (draws) work[base + (int32_t)__popcll(dm & ((1ull << lane) - 1ull))] = k;
  }
  __syncthreads();
  if (tid < nwork) {
    const int32_t kd = work[tid];
    Key k1, k2;
    split2(split_at(Key{a.ck[0], a.ck[1]}, a.n_agents, kd, kMode), k1, k2, kMode);
    const uint32_t j = randint_offset(bits_scalar(k1, kMode), bits_scalar(k2, kMode),
                                      (uint32_t)a.n_empty);
    const int32_t tg = jth_empty(j, empty_prefix_lds, a.nb, a.ebits);
    if (tg >= 0) atomicMin(&a.claim[tg], kd);
    a.target[kd] = tg;
  }
  const uint64_t m = __ballot(happy);
  if ((tid & 63) == 0) wc[tid >> 6] = (int32_t)__popcll(m);
  __syncthreads();
  if (tid == 0) {
    int32_t s = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += wc[w];
    if (s) atomicAdd(a.happy_count, s);
  }
}

// One thread per agent; large workgroups keep the grid small, which is most of
// the cost of a step that only checks the identity condition.  Bound by its
// chain of loads (the identity word and the target, then the claim, the old
// cell and the type, together) and by the drain of its scattered atomics: 7.5 ->
// 5 us in the middle steps at 512 x 512 from two round trips more.
constexpr int kMovesThreads = 1024;

struct SchellingMoves {
  int64_t n_agents;
  int8_t *cells;
  int32_t *id, *claim, *pos;
  const int8_t *type;
  const int32_t *target;
  uint32_t *ebits;
  int32_t *ecount;
  int32_t nb;
  int32_t *moves;
  const int32_t *prev_happy;
};

__global__ void __launch_bounds__(kMovesThreads) k_schelling_moves(SchellingMoves a) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t tg = k < a.n_agents ? a.target[k] : -1;
  if (schelling_identity(a.prev_happy, a.n_agents)) return;  // grid-uniform: no move
  bool moved = false;
  if (tg >= 0) {
    const int32_t winner = a.claim[tg], old = a.pos[k];
    const int8_t type = a.type[k];
    if (winner == (int32_t)k) {
      a.cells[old] = 0;
      a.id[old] = -1;
      a.cells[tg] = type;
      a.id[tg] = (int32_t)k;
      a.pos[k] = tg;
      a.claim[tg] = INT_MAX;
      // the old cell becomes empty, the target occupied (distinct cells: a
      // target was empty before the step, an old cell occupied)
      atomicOr(&a.ebits[old >> 5], 1u << (old & 31));
      atomicAnd(&a.ebits[tg >> 5], ~(1u << (tg & 31)));
      const int32_t bo = old / kCellsPerBlock, bt = tg / kCellsPerBlock;
      if (bo != bt) {
        int32_t *copy = a.ecount + (int64_t)(blockIdx.x % kCountCopies) * a.nb;
        atomicAdd(&copy[bo], 1);
        atomicSub(&copy[bt], 1);
      }
      moved = true;
    }
  }
  __shared__ int32_t wc[kMovesThreads / 64];
  const uint64_t m = __ballot(moved);
  if ((threadIdx.x & 63) == 0) wc[threadIdx.x >> 6] = (int32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t s = 0;
    for (int w = 0; w < kMovesThreads / 64; ++w) s += wc[w];
    if (s) atomicAdd(a.moves, s);
  }
}

// ---- small grids: a whole run in one launch by one workgroup
//
// The two types as bit planes of whole words per row, agent ids, the empty
// list and its claims in LDS.  A step: the unhappy cells, 32 at a time by
// bitwise counts, and the empty ones; one scan of both counts; both lists; the
// draws of the unhappy agents, on full waves, and their claims; the winners'
// moves.  Four barriers.  The run ends at the first identity step, whose
// record every later step repeats.
//
// Bound by the draws (450 instructions an unhappy agent, on one CU) and by the
// latency of the barriers.  Runs of 80 steps, which settle at 13 to 20: 24 x 24
// cells 141 us, 61 x 90 176, 100 x 100 179, 150 x 150 210, with the two
// launches a step of the kernels above 493, 523, 517 and 527; 12 steps of
// 150 x 150, the least favourable, 184 against 293.  So every grid that the LDS
// holds runs here (about 24,000 cells; the one CU's draws would meet the
// launches at some 60,000).  Happiness by agent from byte cells: 61 x 90 236 us.
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr size_t kSmallLds = 155 * 1024;

struct SchellingSmall {
  int32_t H, W, row_words, n_agents, n_empty, steps;
  int8_t *cells;
  int32_t *id, *pos;
  const uint32_t *keys;  // [steps][2]
  const int32_t *prev;   // counters of the step before, or null
  int32_t *counters;     // [steps][2]
  float *happy_frac;
  int32_t *moves;
};

// LDS: the planes and the unhappy bits u32[3][words], claim u32[n_empty],
// id u16[cells], list u16[n_empty], work and draw u16[n_agents]
size_t schelling_small_lds(int32_t H, int32_t W, int64_t n_agents) {
  const int64_t nc = (int64_t)H * W, words = (int64_t)H * ((W + 31) / 32);
  return (size_t)(12 * words + 6 * (nc - n_agents) + 2 * nc + 4 * n_agents);
}

bool schelling_small(int32_t H, int32_t W, int64_t n_agents) {
  return schelling_small_lds(H, W, n_agents) <= kSmallLds;  // so H * W < 2^16
}

// at_least[i]: bits where at least 2^i of the eight words have theirs set;
// exact[i]: where exactly i have, i < 3
__device__ __forceinline__ void bit_counts(const uint32_t (&x)[8], uint32_t (&at_least)[3],
                                           uint32_t (&exact)[3]) {
  const uint32_t s1 = x[0] ^ x[1] ^ x[2], c1 = (x[0] & x[1]) | (x[2] & (x[0] ^ x[1]));
  const uint32_t s2 = x[3] ^ x[4] ^ x[5], c2 = (x[3] & x[4]) | (x[5] & (x[3] ^ x[4]));
  const uint32_t s3 = x[6] ^ x[7], c3 = x[6] & x[7];
  const uint32_t b0 = s1 ^ s2 ^ s3, c4 = (s1 & s2) | (s3 & (s1 ^ s2));
  const uint32_t t = c1 ^ c2 ^ c3, f1 = (c1 & c2) | (c3 & (c1 ^ c2));
  const uint32_t b1 = t ^ c4, f2 = t & c4;
  at_least[2] = f1 | f2;  // 4 or more
  at_least[1] = at_least[2] | b1;
  at_least[0] = at_least[1] | b0;
  exact[0] = ~at_least[0];
  exact[1] = b0 & ~at_least[1];
  exact[2] = b1 & ~b0 & ~at_least[2];
}

// the unhappy bits of a word.  8 same < 3 (same + other) is 5 same < 3 other:
// no like neighbour and 1 or more others, 1 and 2 or more, 2 and 4 or more (3
// would need 6)
__device__ __forceinline__ uint32_t bit_unhappy(uint32_t one, uint32_t two,
                                                const uint32_t (&x1)[8],
                                                const uint32_t (&x2)[8]) {
  uint32_t least1[3], least2[3], is1[3], is2[3];
  bit_counts(x1, least1, is1);
  bit_counts(x2, least2, is2);
  return (one & ((is1[0] & least2[0]) | (is1[1] & least2[1]) | (is1[2] & least2[2]))) |
         (two & ((is2[0] & least1[0]) | (is2[1] & least1[1]) | (is2[2] & least1[2])));
}

// The eight neighbours' bits of word w of row r on the torus.
__device__ __forceinline__ void bit_neighbours(const uint32_t *plane, int32_t r, int32_t w,
                                               int32_t H, int32_t W, int32_t row_words,
                                               uint32_t (&x)[8]) {
  const int32_t rows[3] = {r ? r - 1 : H - 1, r, r + 1 < H ? r + 1 : 0};
  const int32_t last = row_words - 1, end = (W - 1) & 31;  // the last column's word and bit
  uint32_t *out = x;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const uint32_t *row = plane + rows[q] * row_words;
    const uint32_t mid = row[w];
    const uint32_t from_left = w ? row[w - 1] >> 31 : (row[last] >> end) & 1u;
    const uint32_t from_right = w < last ? row[w + 1] << 31 : (row[0] & 1u) << end;
    *out++ = (mid << 1) | from_left;
    *out++ = (mid >> 1) | from_right;
    if (q != 1) *out++ = mid;
  }
}

template <int kMode>
__global__ void __launch_bounds__(kSmallThreads) k_schelling_small(SchellingSmall a) {
  extern __shared__ uint32_t small_lds[];
  __shared__ uint32_t wsum[kSmallWaves];
  __shared__ int32_t moved_sum[2];  // by step parity
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t W = a.W, nc = a.H * W, na = a.n_agents, ne = a.n_empty;
  const int32_t rw = a.row_words, words = a.H * rw;
  uint32_t *one = small_lds, *two = one + words, *sad = two + words, *claim = sad + words;
  uint16_t *id = reinterpret_cast<uint16_t *>(claim + ne);
  uint16_t *list = id + nc, *work = list + ne, *draw = work + na;
  const uint32_t tail = (W & 31) ? (1u << (W & 31)) - 1 : ~0u;  // columns of a row's last word
  // c / W for c < 2^16: (c + 0.5) / W is 0.5 / W or more from a whole number,
  // its rounding errors are below 2^-6 / W
  const float inv_w = 1.0f / (float)W;
  auto row_of = [&](int32_t c) { return (int32_t)(((float)c + 0.5f) * inv_w); };
  for (int32_t w = tid; w < words; w += kSmallThreads) one[w] = two[w] = 0;
  for (int32_t j = tid; j < ne; j += kSmallThreads) claim[j] = INT_MAX;
  if (tid < 2) moved_sum[tid] = 0;
  __syncthreads();
  for (int32_t c = tid; c < nc; c += kSmallThreads) {
    const int8_t v = a.cells[c];
    id[c] = (uint16_t)a.id[c];
    const int32_t r = row_of(c), col = c - r * W;
    if (v) atomicOr(&(v == 1 ? one : two)[r * rw + (col >> 5)], 1u << (col & 31));
  }
  // words of a thread: neighbouring ones, so that the scan numbers the cells row by row
  const int32_t per = (words + kSmallThreads - 1) / kSmallThreads;
  const int32_t w0 = min(tid * per, words), w1 = min(w0 + per, words);
  int32_t prev_happy = a.prev ? a.prev[0] : -1;
  Key key{a.keys[0], a.keys[1]};
  int32_t t = 0;
  __syncthreads();
  for (; t < a.steps && prev_happy != na; ++t) {  // block-uniform
    const int32_t tn = t + 1 < a.steps ? t + 1 : t;
    const Key ck = key;
    key = Key{a.keys[2 * tn], a.keys[2 * tn + 1]};  // the next step's, on its way meanwhile
    uint32_t count = 0;  // empty cells << 16 | unhappy agents
    for (int32_t w = w0; w < w1; ++w) {
      const int32_t r = w / rw, col = w - r * rw;
      uint32_t x1[8], x2[8];
      bit_neighbours(one, r, col, a.H, W, rw, x1);
      bit_neighbours(two, r, col, a.H, W, rw, x2);
      const uint32_t o = one[w], p = two[w];
      const uint32_t u = bit_unhappy(o, p, x1, x2);
      sad[w] = u;
      const uint32_t e = ~(o | p) & (col == rw - 1 ? tail : ~0u);
      count += (uint32_t)__popc(e) << 16 | (uint32_t)__popc(u);
    }
    uint32_t at = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(at, off);
      if (lane >= off) at += y;
    }
    if (lane == 63) wsum[wave] = at;
    __syncthreads();
    at -= count;
    uint32_t total = 0;
#pragma unroll
    for (int q = 0; q < kSmallWaves; ++q) {
      if (q == wave) at += total;
      total += wsum[q];
    }
    const int32_t unhappy = (int32_t)(total & 0xffffu);
    const int32_t nwork = ne > 0 ? min(unhappy, na) : 0;
    for (int32_t w = w0; w < w1; ++w) {
      const int32_t r = w / rw, col = w - r * rw, c0 = r * W + 32 * col;
      for (uint32_t u = sad[w]; u; u &= u - 1) {
        const uint32_t i = at++ & 0xffffu;
        if (i < (uint32_t)na) work[i] = (uint16_t)(c0 + __ffs(u) - 1);
      }
      for (uint32_t e = ~(one[w] | two[w]) & (col == rw - 1 ? tail : ~0u); e; e &= e - 1) {
        const uint32_t j = at >> 16;
        if (j < (uint32_t)ne) list[j] = (uint16_t)(c0 + __ffs(e) - 1);
        at += 1u << 16;
      }
    }
    __syncthreads();
    // draws and claims (lowest agent wins)
    for (int32_t i = tid; i < nwork; i += kSmallThreads) {
      const uint32_t k = id[work[i]];
      Key k1, k2;
      split2(split_at(ck, na, k, kMode), k1, k2, kMode);
      const uint32_t j = randint_offset(bits_scalar(k1, kMode), bits_scalar(k2, kMode),
                                        (uint32_t)ne);
      draw[i] = (uint16_t)j;
      atomicMin(&claim[j], k);
    }
    if (tid == 0) moved_sum[(t + 1) & 1] = 0;  // last read before this step's first barrier
    __syncthreads();
    // moves: old cells and targets are distinct; a winner frees its claim (a
    // loser that reads it then still loses)
    int32_t moved = 0;
    for (int32_t i = tid; i < nwork; i += kSmallThreads) {
      const int32_t old = work[i], j = draw[i];
      const uint32_t k = id[old];
      if (claim[j] == k) {
        const int32_t to = list[j], r0 = row_of(old), r1 = row_of(to);
        const int32_t col0 = old - r0 * W, col1 = to - r1 * W;
        const int32_t from = r0 * rw + (col0 >> 5), into = r1 * rw + (col1 >> 5);
        const uint32_t bit = 1u << (col0 & 31);
        uint32_t *plane = (one[from] & bit) ? one : two;
        atomicAnd(&plane[from], ~bit);
        atomicOr(&plane[into], 1u << (col1 & 31));
        id[to] = (uint16_t)k;
        claim[j] = INT_MAX;
        ++moved;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) moved += __shfl_xor(moved, off);
    if (lane == 0 && moved) atomicAdd(&moved_sum[t & 1], moved);
    __syncthreads();
    prev_happy = na - unhappy;
    if (tid == 0) {
      const int32_t m = moved_sum[t & 1];
      a.counters[2 * t] = prev_happy;
      a.counters[2 * t + 1] = m;
      a.happy_frac[t] = (float)prev_happy / (float)(na > 0 ? na : 1);
      a.moves[t] = m;
    }
  }
  for (int32_t u = t + tid; u < a.steps; u += kSmallThreads) {  // identity steps
    a.counters[2 * u] = na;
    a.counters[2 * u + 1] = 0;
    a.happy_frac[u] = (float)na / (float)(na > 0 ? na : 1);
    a.moves[u] = 0;
  }
  if (t == 0) return;
  for (int32_t c = tid; c < nc; c += kSmallThreads) {
    const int32_t r = row_of(c), col = c - r * W, w = r * rw + (col >> 5), b = col & 31;
    const int8_t v = (int8_t)((one[w] >> b & 1u) + 2 * (two[w] >> b & 1u));
    a.cells[c] = v;
    a.id[c] = v ? id[c] : -1;
    if (v) a.pos[id[c]] = c;
  }
}

// record[t] = (happy fraction, moves) from the integer counters; the steps from
// `launched` on are the identity and get their counters here
__global__ void k_schelling_record(int32_t *__restrict__ counters, int32_t steps,
                                   int32_t launched, int64_t n_agents,
                                   float *__restrict__ happy_frac, int32_t *__restrict__ moves) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= steps) return;
  if (t >= launched) counters[2 * t] = (int32_t)n_agents;
  happy_frac[t] = (float)counters[2 * t] / (float)(n_agents > 0 ? n_agents : 1);
  moves[t] = counters[2 * t + 1];
}

// settled steps: each is the identity when the step before them found every
// agent happy; otherwise the records are marked invalid (-1, NaN, -1)
__global__ void k_schelling_settled(const int32_t *__restrict__ prev_counters, int32_t steps,
                                    int64_t n_agents, int32_t *__restrict__ counters,
                                    float *__restrict__ happy_frac,
                                    int32_t *__restrict__ moves) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= steps) return;
  const bool ok = (int64_t)prev_counters[0] == n_agents;
  counters[2 * t] = ok ? (int32_t)n_agents : -1;
  counters[2 * t + 1] = ok ? 0 : -1;
  happy_frac[t] = ok ? (float)n_agents / (float)(n_agents > 0 ? n_agents : 1)
                     : __int_as_float(0x7fc00000);
  moves[t] = ok ? 0 : -1;
}

__global__ void k_schelling_init_cells(const uint32_t *__restrict__ key, int64_t nc,
                                       int8_t *__restrict__ cells, int32_t *__restrict__ claim,
                                       int mode) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const float u = unit_float(bits_at(Key{key[0], key[1]}, nc, c, mode));
  cells[c] = u < 0.45f ? 1 : (u < 0.9f ? 2 : 0);
  claim[c] = INT_MAX;
}

__global__ void k_fill_i32_s(int32_t *__restrict__ p, int64_t n, int32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// k_schelling_small may need more than 64 KB of dynamic LDS: the limit is
// raised once per device, under a lock.
constexpr int kMaxDevices = 64;
std::mutex g_schelling_attr_mu;
bool g_schelling_attr_set[kMaxDevices];

int schelling_lds_attr() {
  int dev = -1;
  ABM_CHECK_HIP(hipGetDevice(&dev));
  ABM_REQUIRE(dev >= 0 && dev < kMaxDevices, "schelling: device index out of range");
  std::lock_guard<std::mutex> lock(g_schelling_attr_mu);
  if (!g_schelling_attr_set[dev]) {
    for (const void *k : {(const void *)k_schelling_small<kModeOriginal>,
                          (const void *)k_schelling_small<kModePartitionable>})
      ABM_CHECK_HIP(
          hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds));
    g_schelling_attr_set[dev] = true;
  }
  return kOk;
}

inline unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

int check_grid(const abm_schelling_grid *g, const char *who) {
  if (!g || g->height < 1 || g->width < 1 ||
      (int64_t)g->height * g->width >= (1ll << 31) || !g->cells || !g->id || !g->claim ||
      !g->pos || !g->type || !g->target || !g->empty || !g->block_counts ||
      g->n_agents < 0 || g->n_agents > (int64_t)g->height * g->width) {
    set_error(std::string(who) + ": bad grid descriptor");
    return kErrInvalid;
  }
  return kOk;
}

}  // namespace abm

using namespace abm;

extern "C" {

int64_t abm_schelling_block_count(int64_t n_cells) {
  return kCountCopies * ((n_cells + kCellsPerBlock - 1) / kCellsPerBlock);
}

int abm_schelling_one_launch(const abm_schelling_grid *g) {
  if (check_grid(g, "abm_schelling_one_launch")) return 0;
  return schelling_small(g->height, g->width, g->n_agents) ? 1 : 0;
}

int abm_schelling_init(abm_schelling_grid *g, const uint32_t *key, int mode,
                       int32_t *n_agents_out, void *stream) {
  if (!g || g->height < 1 || g->width < 1) {
    set_error("abm_schelling_init: bad grid");
    return kErrInvalid;
  }
  ABM_REQUIRE(key && n_agents_out && (mode == 0 || mode == 1),
              "abm_schelling_init: bad arguments");
  const int64_t nc = (int64_t)g->height * g->width;
  g->n_agents = 0;
  if (int rc = check_grid(g, "abm_schelling_init")) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_schelling_init_cells, dim3(nblk(nc, 256)), dim3(256), 0, s, key, nc,
                     g->cells, g->claim, mode);
  const unsigned nb = nblk(nc, kCellsPerBlock);
  hipLaunchKernelGGL(k_cells_count, dim3(nb), dim3(kCellsPerBlock), 0, s, g->cells, nc, 0,
                     g->block_counts);
  hipLaunchKernelGGL(k_cells_scatter, dim3(nb), dim3(kCellsPerBlock), 0, s, g->cells, nc, 0,
                     g->block_counts, g->pos, g->type, g->id);
  ABM_LAUNCH_CHECK("abm_schelling_init");
  // agent count: sum of the block counts (host read; set-up only)
  int32_t *host = new int32_t[nb];
  hipError_t e = hipMemcpyAsync(host, g->block_counts, nb * sizeof(int32_t),
                                hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    delete[] host;
    return hip_fail(e, "abm_schelling_init");
  }
  int64_t na = 0;
  for (unsigned b = 0; b < nb; ++b) na += host[b];
  delete[] host;
  g->n_agents = na;
  *n_agents_out = (int32_t)na;
  return kOk;
}

}  // extern "C"

// A watched run learns from the agents kernels how far it is; each
// kWatchEvery-th step tells, and up to twice as many identity steps follow the
// last move: 28 of 200 steps launched at 512 x 512, where 23 move or look, against
// 48 in launches of 16 steps.  A run 648 us before, 484 with this and the kernels'
// single round of loads.
constexpr int32_t kWatchEvery = 4;

// the step loop of a run; prev0: the counters of the step before the first
// (nullptr: a fresh run, whose bitmap and block counts are built from the cells
// first); watch: launching stops once a step was the identity
static int schelling_steps(const abm_schelling_grid *g, const uint32_t *keys, int32_t steps,
                           int mode, const int32_t *prev0, int32_t *counters, float *happy_frac,
                           int32_t *moves, int32_t *watch, int32_t *launched, void *stream,
                           const char *what) {
  if (int rc = check_grid(g, what)) return rc;
  ABM_REQUIRE(keys && counters && happy_frac && moves && steps >= 0 &&
                  (mode == 0 || mode == 1),
              "abm_schelling_run: bad arguments");
  if (launched) *launched = steps;
  if (steps == 0) return kOk;
  hipStream_t s = (hipStream_t)stream;
  const int64_t nc = (int64_t)g->height * g->width;
  const int64_t n_empty = nc - g->n_agents;
  const unsigned nb = nblk(nc, kCellsPerBlock);
  ABM_REQUIRE(nb <= kMaxEmptyBlocks,
              "abm_schelling_run: grids of more than 15,360,000 cells are not supported");
  // the bitmap's lines are read 16 bytes at a time, so it begins at the first
  // such boundary of the scratch; whole blocks of words fit from there: 32 * nb + 3
  // <= H*W for any grid not run below
  uint32_t *ebits = reinterpret_cast<uint32_t *>(((uintptr_t)g->empty + 15u) & ~(uintptr_t)15u);
  const bool part = mode == kModePartitionable;
  if (schelling_small(g->height, g->width, g->n_agents)) {
    if (int rc = schelling_lds_attr()) return rc;
    SchellingSmall a;
    a.H = g->height;
    a.W = g->width;
    a.row_words = (a.W + 31) / 32;
    a.n_agents = (int32_t)g->n_agents;
    a.n_empty = (int32_t)n_empty;
    a.steps = steps;
    a.cells = g->cells;
    a.id = g->id;
    a.pos = g->pos;
    a.keys = keys;
    a.prev = prev0;
    a.counters = counters;
    a.happy_frac = happy_frac;
    a.moves = moves;
    hipLaunchKernelGGL(part ? k_schelling_small<kModePartitionable>
                            : k_schelling_small<kModeOriginal>,
                       dim3(1), dim3(kSmallThreads),
                       schelling_small_lds(g->height, g->width, g->n_agents), s, a);
    ABM_LAUNCH_CHECK(what);
    return kOk;
  }
  if (steps <= 2 * kWatchEvery) watch = nullptr;  // too short to stop: no step tells
  if (watch) clear_watch(watch);
  hipLaunchKernelGGL(k_fill_i32_s, dim3(nblk(2 * (int64_t)steps, 256)), dim3(256), 0, s,
                     counters, 2 * (int64_t)steps, 0);
  if (!prev0) {
    hipLaunchKernelGGL(k_empty_bits, dim3(nb), dim3(kCellsPerBlock), 0, s, g->cells, nc, ebits);
    // copy 0 = the grid's empty counts, the other copies start at zero
    hipLaunchKernelGGL(k_cells_count, dim3(nb), dim3(kCellsPerBlock), 0, s, g->cells, nc, 1,
                       g->block_counts);
    const int64_t zero_words = (int64_t)(kCountCopies - 1) * nb;
    hipLaunchKernelGGL(k_fill_i32_s, dim3(nblk(zero_words, 256)), dim3(256), 0, s,
                       g->block_counts + nb, zero_words, 0);
  }
  const dim3 tiles((unsigned)((g->width + kTileDim - 1) / kTileDim),
                   (unsigned)((g->height + kTileDim - 1) / kTileDim));
  const size_t prefix_lds = (size_t)(nb + 1) * sizeof(int32_t);
  int32_t t = 0;
  for (; t < steps; ++t) {
    const bool tells = watch && t % kWatchEvery == 0;
    if (tells && t >= 2 * kWatchEvery) {
      bool settled = false;
      if (int rc = wait_begun(watch, t + 1 - kWatchEvery, s, what, &settled)) return rc;
      if (settled) break;
    }
    const int32_t *prev = t ? counters + 2 * (int64_t)(t - 1) : prev0;
    SchellingStep a;
    a.H = g->height;
    a.W = g->width;
    a.n_agents = g->n_agents;
    a.n_empty = n_empty;
    a.cells = g->cells;
    a.id = g->id;
    a.ebits = ebits;
    a.ecount = g->block_counts;
    a.nb = (int32_t)nb;
    a.claim = g->claim;
    a.target = g->target;
    a.ck = keys + 2 * (int64_t)t;
    a.happy_count = counters + 2 * (int64_t)t;
    a.prev_happy = prev;
    a.watch = watch;
    a.begun = tells ? t + 1 : 0;
    hipLaunchKernelGGL(part ? k_schelling_agents<kModePartitionable>
                            : k_schelling_agents<kModeOriginal>,
                       tiles, dim3(kTileDim * kTileDim), prefix_lds, s, a);
    if (g->n_agents > 0) {
      SchellingMoves m;
      m.n_agents = g->n_agents;
      m.cells = g->cells;
      m.id = g->id;
      m.claim = g->claim;
      m.pos = g->pos;
      m.type = g->type;
      m.target = g->target;
      m.ebits = ebits;
      m.ecount = g->block_counts;
      m.nb = (int32_t)nb;
      m.moves = counters + 2 * (int64_t)t + 1;
      m.prev_happy = prev;
      hipLaunchKernelGGL(k_schelling_moves, dim3(nblk(g->n_agents, kMovesThreads)),
                         dim3(kMovesThreads), 0, s, m);
    }
  }
  hipLaunchKernelGGL(k_schelling_record, dim3(nblk(steps, 256)), dim3(256), 0, s, counters,
                     steps, t, g->n_agents, happy_frac, moves);
  if (launched) *launched = t;
  ABM_LAUNCH_CHECK(what);
  return kOk;
}

extern "C" {

int abm_schelling_run(const abm_schelling_grid *g, const uint32_t *keys, int32_t steps,
                      int mode, int32_t *counters, float *happy_frac, int32_t *moves,
                      void *stream) {
  return schelling_steps(g, keys, steps, mode, nullptr, counters, happy_frac, moves, nullptr,
                         nullptr, stream, "abm_schelling_run");
}

int abm_schelling_run_from(const abm_schelling_grid *g, const uint32_t *keys, int32_t steps,
                           int mode, const int32_t *prev_counters, int32_t *counters,
                           float *happy_frac, int32_t *moves, void *stream) {
  ABM_REQUIRE(prev_counters, "abm_schelling_run_from: prev_counters is null");
  return schelling_steps(g, keys, steps, mode, prev_counters, counters, happy_frac, moves,
                         nullptr, nullptr, stream, "abm_schelling_run_from");
}

int abm_schelling_run_watched(const abm_schelling_grid *g, const uint32_t *keys, int32_t steps,
                              int mode, const int32_t *prev_counters, int32_t *counters,
                              float *happy_frac, int32_t *moves, int32_t *watch,
                              int32_t *launched, void *stream) {
  ABM_REQUIRE(watch && launched, "abm_schelling_run_watched: null buffer");
  return schelling_steps(g, keys, steps, mode, prev_counters, counters, happy_frac, moves, watch,
                         launched, stream, "abm_schelling_run_watched");
}

int abm_schelling_settled(const abm_schelling_grid *g, const int32_t *prev_counters, int32_t steps,
                          int32_t *counters, float *happy_frac, int32_t *moves, void *stream) {
  if (int rc = check_grid(g, "abm_schelling_settled")) return rc;
  ABM_REQUIRE(prev_counters && counters && happy_frac && moves && steps >= 0,
              "abm_schelling_settled: bad arguments");
  if (steps == 0) return kOk;
  hipLaunchKernelGGL(k_schelling_settled, dim3(nblk(steps, 256)), dim3(256), 0,
                     (hipStream_t)stream, prev_counters, steps, g->n_agents, counters, happy_frac,
                     moves);
  ABM_LAUNCH_CHECK("abm_schelling_settled");
  return kOk;
}

}  // extern "C"
