// sort.hip -- stable LSD radix sort of (uint32 key, int32 value) pairs and
// jax.random.permutation built on it.
//
// jax.random.permutation(key, n) (reference call sites
// jaxabm/analysis.py:87 and the Deffuant/SIR programs' pairing and seeding)
// runs ceil(3 ln n / ln(2^32-1)) rounds of: key, sub = split(key);
// x = sort_key_val(bits(sub, (n,)), x) with a STABLE sort, so ties among the
// 32-bit keys keep their previous order.  Ties are likely at n = 65,536
// (birthday bound), so the sort must be stable: an LSD radix sort whose
// per-tile ranks follow the input order is.
//
// Per 8-bit digit pass: (1) tile histograms, (2) per digit, an exclusive scan
// of its tile counts and their total, (3) stable scatter: each tile scans the
// 256 totals itself, and ranks within a 64-wide wavefront by ballot matching
// on the digit bits.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.hpp"
#include "jaxabm_amd.h"

namespace abm {

constexpr int kSortThreads = 256;
constexpr int kSortRounds = 8;  // items per thread per tile, in rounds
constexpr int kTile = kSortThreads * kSortRounds;
constexpr int kWaves = kSortThreads / 64;

__global__ void __launch_bounds__(kSortThreads)
    k_digit_hist(const uint32_t *__restrict__ keys, int64_t n, int shift,
                 uint32_t *__restrict__ hist, int tiles) {
  // segment blockIdx.y: keys[seg * n ..), hist[seg * 256 * tiles ..)
  keys += (int64_t)blockIdx.y * n;
  hist += (int64_t)blockIdx.y * 256 * tiles;
  __shared__ uint32_t cnt[256];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kTile + threadIdx.x;
  uint32_t key[kSortRounds];  // all loads in flight
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const int64_t i = base + r * kSortThreads;
    key[r] = keys[i < n ? i : n - 1];
  }
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
    if (base + r * kSortThreads < n) atomicAdd(&cnt[(key[r] >> shift) & 255u], 1u);
  __syncthreads();
  hist[(int64_t)threadIdx.x * tiles + blockIdx.x] = cnt[threadIdx.x];
}

// In place: digit row d = hist[d * tiles ..) becomes its exclusive scan, its
// sum goes to totals[d]; one wavefront per digit, 64 x kScanLoads counts per
// round.  The scan across digits is left to the scatter (256 values).  Bound
// by the round's load latency.  One workgroup scanning all 256 * tiles counts
// (each thread a contiguous, uncoalesced run) took 107 us a pass at 1,000,000
// keys, five times the scatter; this takes 4.
constexpr int kScanLoads = 4;

__global__ void __launch_bounds__(kSortThreads)
    k_digit_scan(uint32_t *__restrict__ hist, int tiles, uint32_t *__restrict__ totals) {
  const int lane = threadIdx.x & 63;
  const int d = blockIdx.x * kWaves + (threadIdx.x >> 6);
  uint32_t *row = hist + ((int64_t)blockIdx.y * 256 + d) * tiles;
  uint32_t run = 0;
  for (int64_t b = 0; b < tiles; b += 64 * kScanLoads) {
    uint32_t v[kScanLoads];
#pragma unroll
    for (int k = 0; k < kScanLoads; ++k) {
      const int64_t i = b + k * 64 + lane;
      v[k] = i < tiles ? row[i] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kScanLoads; ++k) {
      const int64_t i = b + k * 64 + lane;
      uint32_t inc = v[k];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(inc, off);
        if (lane >= off) inc += y;
      }
      if (i < tiles) row[i] = run + inc - v[k];
      run += __shfl(inc, 63);
    }
  }
  if (lane == 0) totals[(int64_t)blockIdx.y * 256 + d] = run;
}

// The same with one workgroup a segment, for at most G tiles: G lanes a digit,
// so that a load covers whole lines and all loads are in flight at once.  With
// 64 workgroups a segment, 200 segments of 2,000 keys spent 18 us of a 29 us
// pass on launching them, and one workgroup with a thread a digit took as long
// at 32 tiles, on its scattered loads.
template <int G>
struct FewTiles {
  static constexpr int kThreads = G < 4 ? 256 * G : 1024;
  static constexpr int kRounds = 256 * G / kThreads;
};

template <int G>
__global__ void __launch_bounds__(FewTiles<G>::kThreads)
    k_digit_scan_few(uint32_t *__restrict__ hist, int tiles, uint32_t *__restrict__ totals) {
  constexpr int T = FewTiles<G>::kThreads, R = FewTiles<G>::kRounds;
  const int place = threadIdx.x & (G - 1);
  hist += (int64_t)blockIdx.x * 256 * tiles;
  totals += (int64_t)blockIdx.x * 256;
  uint32_t v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = (r * T + (int)threadIdx.x) / G;
    v[r] = place < tiles ? hist[d * tiles + place] : 0u;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = (r * T + (int)threadIdx.x) / G;
    uint32_t inc = v[r];
#pragma unroll
    for (int off = 1; off < G; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off);
      if (place >= off) inc += y;
    }
    if (place < tiles) hist[d * tiles + place] = inc - v[r];
    if (place == G - 1) totals[d] = inc;
  }
}

// Tiles up to which one workgroup scans a segment, and up to which it does for
// few segments, where spreading it is faster (one permutation of 65,536, 32
// tiles: 102 us spread and 114; 32 of them: 421 and 420; 200: 2,270 and 2,176).
constexpr int kFewTiles = 32, kFewTilesAlone = 16;
constexpr int64_t kFewSegments = 16;

void digit_scan(uint32_t *hist, int tiles, uint32_t *totals, int64_t segs, hipStream_t s) {
  auto few = [&](auto g) {
    constexpr int G = decltype(g)::value;
    hipLaunchKernelGGL(k_digit_scan_few<G>, dim3((unsigned)segs), dim3(FewTiles<G>::kThreads), 0,
                       s, hist, tiles, totals);
  };
  if (tiles > (segs < kFewSegments ? kFewTilesAlone : kFewTiles))
    hipLaunchKernelGGL(k_digit_scan, dim3(256 / kWaves, (unsigned)segs), dim3(kSortThreads), 0, s,
                       hist, tiles, totals);
  else if (tiles > 16)
    few(std::integral_constant<int, 32>{});
  else if (tiles > 4)
    few(std::integral_constant<int, 16>{});
  else if (tiles > 1)
    few(std::integral_constant<int, 4>{});
  else
    few(std::integral_constant<int, 1>{});
}

// Stable scatter of one digit.  Wave w of tile b owns items [b kTile + w 64
// kSortRounds, ..) of the segment, 64 per round, so wave order and round order
// are input order.  The loads of all rounds are issued together; each wave
// counts its digits (LDS atomics), one pass over the waves turns the counts
// into each wave's first position per digit, and from there a wave ranks and
// stores its rounds alone: three barriers a tile instead of four a round, with
// one load latency instead of one per round (1,000,000 pairs: 18.8 -> 16.7 us;
// what is left is the scattered 4-byte stores).
__global__ void __launch_bounds__(kSortThreads)
    k_digit_scatter(const uint32_t *__restrict__ keys_in,
                    const int32_t *__restrict__ vals_in, int64_t n, int shift,
                    const uint32_t *__restrict__ offsets,
                    const uint32_t *__restrict__ totals, int tiles,
                    uint32_t *__restrict__ keys_out,
                    int32_t *__restrict__ vals_out) {
  {
    const int64_t seg = (int64_t)blockIdx.y * n;
    keys_in += seg;
    vals_in += seg;
    keys_out += seg;
    vals_out += seg;
    offsets += (int64_t)blockIdx.y * 256 * tiles;
    totals += (int64_t)blockIdx.y * 256;
  }
  __shared__ uint32_t wpos[kWaves][256];
  __shared__ uint32_t wsum[kWaves];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t first = (int64_t)blockIdx.x * kTile + (int64_t)wave * 64 * kSortRounds + lane;
  uint32_t key[kSortRounds];
  int32_t val[kSortRounds];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const int64_t i = first + r * 64;
    key[r] = i < n ? keys_in[i] : 0u;
    val[r] = i < n ? vals_in[i] : 0;
  }
  const uint32_t own = offsets[(int64_t)t * tiles + blockIdx.x];
  const uint32_t total = totals[t];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) wpos[w][t] = 0;
  uint32_t inc = total;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(inc, off);
    if (lane >= off) inc += y;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
    if (first + r * 64 < n) atomicAdd(&wpos[wave][(key[r] >> shift) & 255u], 1u);
  // digit base: the keys of smaller digits, then this digit's earlier tiles
  uint32_t pos = own + inc - total;
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    if (w < wave) pos += wsum[w];
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t c = wpos[w][t];
    wpos[w][t] = pos;
    pos += c;
  }
  __syncthreads();
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  volatile uint32_t *mine = wpos[wave];  // this wave's alone from here on
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const bool valid = first + r * 64 < n;
    const uint32_t d = (key[r] >> shift) & 255u;
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    if (valid) {
      const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
      const uint32_t at = mine[d];
      // LDS operations of a wave complete in order: every lane has read the
      // digit's position before its first lane moves it on
      __builtin_amdgcn_wave_barrier();
      if (rank == 0) mine[d] = at + (uint32_t)__popcll(peers);
      keys_out[at + rank] = key[r];
      vals_out[at + rank] = val[r];
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// out[s * n + i] = i for segment s = blockIdx.y
__global__ void k_iota(int32_t *__restrict__ out, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[(int64_t)blockIdx.y * n + i] = (int32_t)i;
}

// Round r's sort keys: k_0 = key; k_{j+1}, sub_j = split(k_j); bits(sub_r).
// Segment s = blockIdx.y takes its key at key[s * key_stride].
// Round 0 also writes the identity the sorts permute, iota[s * n + i] = i.
__global__ void k_perm_round_bits(const uint32_t *__restrict__ key, int64_t key_stride,
                                  int round, int64_t n, uint32_t *__restrict__ out,
                                  int32_t *__restrict__ iota, int mode) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  key += (int64_t)blockIdx.y * key_stride;
  out += (int64_t)blockIdx.y * n;
  Key k{key[0], key[1]}, sub;
  for (int j = 0; j <= round; ++j) {
    Key nk;
    split2(k, nk, sub, mode);
    k = nk;
  }
  out[i] = bits_at(sub, n, i, mode);
  if (round == 0) iota[(int64_t)blockIdx.y * n + i] = (int32_t)i;
}

size_t sort_workspace_bytes(int64_t n, int64_t segs = 1) {
  int64_t tiles = (n + kTile - 1) / kTile;
  // the second key and value buffers, tile histograms, digit totals
  size_t b = 0;
  b += (size_t)n * (size_t)segs * 4 * 2;
  b += (size_t)tiles * 256 * 4 * (size_t)segs;
  b += (size_t)256 * 4 * (size_t)segs;
  return (b + 255) & ~(size_t)255;
}

// Sort each of `segs` consecutive segments of n (key, value) pairs, keys[]
// destroyed, vals[] in place, using ws.
int radix_sort_pairs(uint32_t *keys, int32_t *vals, int64_t n, void *ws,
                     hipStream_t s, int64_t segs = 1) {
  if (n <= 1 || segs < 1) return kOk;
  int tiles = (int)((n + kTile - 1) / kTile);
  const int64_t total = n * segs;
  char *p = (char *)ws;
  uint32_t *k2 = (uint32_t *)p;
  p += (size_t)total * 4;
  int32_t *v2 = (int32_t *)p;
  p += (size_t)total * 4;
  uint32_t *hist = (uint32_t *)p;
  p += (size_t)tiles * 256 * 4 * (size_t)segs;
  uint32_t *totals = (uint32_t *)p;
  uint32_t *ka = keys, *kb = k2;
  int32_t *va = vals, *vb = v2;
  const dim3 grid((unsigned)tiles, (unsigned)segs);
  for (int shift = 0; shift < 32; shift += 8) {
    hipLaunchKernelGGL(k_digit_hist, grid, dim3(kSortThreads), 0, s, ka, n, shift, hist,
                       tiles);
    digit_scan(hist, tiles, totals, segs, s);
    hipLaunchKernelGGL(k_digit_scatter, grid, dim3(kSortThreads), 0, s, ka, va, n, shift,
                       hist, (const uint32_t *)totals, tiles, kb, vb);
    uint32_t *tk = ka;
    ka = kb;
    kb = tk;
    int32_t *tv = va;
    va = vb;
    vb = tv;
  }
  // 4 passes: the result is back in (keys, vals)
  ABM_LAUNCH_CHECK("radix_sort_pairs");
  return kOk;
}

// permutation(key_s, n) for segs keys (key_s at keys[s * key_stride]), the
// results in out[s * n ..).
int permutation_segments(const uint32_t *keys, int64_t key_stride, int64_t segs, int64_t n,
                         int32_t *out, void *ws, int mode, hipStream_t s) {
  const dim3 g((unsigned)((n + 255) / 256), (unsigned)segs);
  uint32_t *bits = (uint32_t *)((char *)ws + sort_workspace_bytes(n, segs));
  const int rounds = (int)__builtin_ceil(3.0 * __builtin_log((double)(n > 1 ? n : 1)) /
                                         __builtin_log(4294967295.0));
  if (rounds == 0)  // n == 1
    hipLaunchKernelGGL(k_iota, g, dim3(256), 0, s, out, n);
  for (int r = 0; r < rounds; ++r) {
    hipLaunchKernelGGL(k_perm_round_bits, g, dim3(256), 0, s, keys, key_stride, r, n, bits,
                       out, mode);
    int rc = radix_sort_pairs(bits, out, n, ws, s, segs);
    if (rc) return rc;
  }
  return kOk;
}

}  // namespace abm

using namespace abm;

extern "C" {

size_t abm_permutation_workspace(int64_t n) {
  return sort_workspace_bytes(n) + (((size_t)n * 4 + 255) & ~(size_t)255);
}

int abm_permutation_rounds(int64_t n) {
  double nn = (double)(n > 1 ? n : 1);
  return (int)__builtin_ceil(3.0 * __builtin_log(nn) / __builtin_log(4294967295.0));
}

int abm_permutation(const uint32_t *key, int64_t n, int32_t *out, void *ws,
                    size_t ws_bytes, int mode, void *stream) {
  ABM_REQUIRE(n >= 0 && n < (1ll << 31), "abm_permutation: n out of range");
  ABM_REQUIRE(mode == 0 || mode == 1, "abm_permutation: bad mode");
  if (n == 0) return kOk;
  ABM_REQUIRE(key && out && ws && ws_bytes >= abm_permutation_workspace(n),
              "abm_permutation: workspace too small");
  int rc = permutation_segments(key, 0, 1, n, out, ws, mode, (hipStream_t)stream);
  if (rc) return rc;
  ABM_LAUNCH_CHECK("abm_permutation");
  return kOk;
}

size_t abm_permutation_batch_workspace(int64_t n, int32_t count) {
  if (n < 0 || count < 0) return 0;
  return sort_workspace_bytes(n, count) +
         (((size_t)n * (size_t)count * 4 + 255) & ~(size_t)255);
}

int abm_permutation_batch(const uint32_t *keys, int64_t key_stride, int32_t count, int64_t n,
                          int32_t *out, void *ws, size_t ws_bytes, int mode, void *stream) {
  ABM_REQUIRE(n >= 0 && n < (1ll << 31) && count >= 0 && count < 65536 &&
                  n * (int64_t)count < (1ll << 31) && key_stride >= 2,
              "abm_permutation_batch: sizes out of range");
  ABM_REQUIRE(mode == 0 || mode == 1, "abm_permutation_batch: bad mode");
  if (n == 0 || count == 0) return kOk;
  ABM_REQUIRE(keys && out && ws && ws_bytes >= abm_permutation_batch_workspace(n, count),
              "abm_permutation_batch: workspace too small");
  int rc = permutation_segments(keys, key_stride, count, n, out, ws, mode, (hipStream_t)stream);
  if (rc) return rc;
  ABM_LAUNCH_CHECK("abm_permutation_batch");
  return kOk;
}

int abm_sort_pairs_u32(uint32_t *keys, int32_t *vals, int64_t n, void *ws,
                       size_t ws_bytes, void *stream) {
  ABM_REQUIRE(n >= 0 && n < (1ll << 31), "abm_sort_pairs_u32: n out of range");
  if (n <= 1) return kOk;
  ABM_REQUIRE(ws && ws_bytes >= sort_workspace_bytes(n),
              "abm_sort_pairs_u32: workspace too small");
  return radix_sort_pairs(keys, vals, n, ws, (hipStream_t)stream);
}

}  // extern "C"
