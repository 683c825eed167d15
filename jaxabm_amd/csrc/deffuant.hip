// deffuant.hip -- differentiable Deffuant bounded-confidence model: batched
// forward step, final statistics and loss, and the hand-written adjoint with
// checkpointed recomputation.
//
// Program (reference API: one collection, env-phase pairing with the update
// key, jaxabm/model.py:146-216; loss and gradient set-up
// jaxabm/analysis.py:489-531):
//  init   agent keys = split(init_key, n); x_i = uniform(agent_key_i), the
//         same value for every instance of the batch
//  step   perm = permutation(uk, n), shared by the batch (common random
//         numbers); pairs (perm[2i], perm[2i+1]); d = x_c - x_a;
//         g = 1 / (1 + exp(-(eps - |d|) / 0.02)); delta = (mu g) d;
//         x_a += delta; x_c -= delta (an odd agent out keeps its opinion)
//  loss   stats = [mean, variance, 32-bin soft histogram with edges k/32,
//         bin k = mean sigmoid(128 (x - k/32)) - sigmoid(128 (x - (k+1)/32))];
//         L = sum (stats - target)^2 per instance, in float64
//
// Layout (HBM): x[n][B], agent-major and instance-minor, so a pair reads and
// writes two contiguous rows of B floats: every access is a coalesced row
// segment whatever the pairing.  In the step kernels the 64 lanes of a
// wavefront span VEC-wide column groups and the waves span pairs.
//
// Adjoint of one step, per pair and instance (lam = dL/dx after the step):
//   g' = g (1 - g) / 0.02
//   fd = d delta/dd   = mu (g - |d| g')     w = lam_a - lam_c
//   fe = d delta/deps = mu d g'             lam_a -= w fd, lam_c += w fd
//   fm = d delta/dmu  = g d                 dL/deps += w fe, dL/dmu += w fm
// The parameter sums are float64; each workgroup row of the grid owns one
// accumulator slot for the whole sweep (same slot every step), and the slots
// are summed in a fixed order, so the gradients are deterministic.
// Checkpoints: the forward keeps the state at every ckpt_every-th step; the
// backward recomputes each segment's states from its checkpoint, then sweeps
// the segment in reverse.
//
// Column runs (ABM_DEFFUANT_COLUMNS): the instances never meet, so one
// workgroup can keep the opinions of one instance in LDS and run all its
// steps in one launch, where the step kernels above read and write the whole
// batch once per step.  See "column runs" below.
#include <hip/hip_runtime.h>

#include <mutex>

#include "common.hpp"
#include "deffuant_gate.hpp"
#include "jaxabm_amd.h"

namespace abm {

constexpr int kDefThreads = 256;
constexpr int kDefWaves = kDefThreads / 64;
// most row chunks of the statistics: two wavefronts per SIMD at 256 columns,
// and eight rounds of loads to sum them
constexpr int64_t kStatChunks = 512;
constexpr int kStatLen = 2 + 32;
constexpr int kHistBins = 32;
constexpr double kHistSlope = 128.0;

template <int VEC>
__device__ __forceinline__ void load_cols(const float *p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const float4 t = *reinterpret_cast<const float4 *>(p);
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
  } else {
    v[0] = *p;
  }
}

template <int VEC>
__device__ __forceinline__ void store_cols(float *p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    *p = v[0];
  }
}

// The gates of P differences, the same bits as gate(): the short form, 34
// operations a gate instead of about 58, unless an argument of the wavefront is
// outside its range or NaN.  eps(u): the bound of difference u.
template <int P, class Eps>
__device__ __forceinline__ void gates(Eps eps, const float (&d)[P], float (&g)[P]) {
  bool odd = false;
#pragma unroll
  for (int u = 0; u < P; ++u) {
    const float num = eps(u) - fabsf(d[u]);
    odd |= !(fabsf(num) <= kGateShort);
    // within 1 ulp, and rounded where inv_rounded asks for it
    g[u] = gate_short(num, [](float x) { return __builtin_amdgcn_rcpf(x); });
  }
  if (__ballot(odd)) {
#pragma unroll
    for (int u = 0; u < P; ++u) g[u] = gate(eps(u), d[u]);
  }
}

// Pairs each wavefront holds in flight per loop iteration of the step kernel:
// eight 1 KB row loads outstanding per wave (measured: 4 beats 2 and 8).
constexpr int kDefStepPairs = 4;

// One step for the whole batch.  Bound by the 128 MB a step moves at 65,536 x
// 256 (23 us a step with gates(), 25.7 with gate()).  src == dst updates in place (pairs are
// disjoint); otherwise every row of dst is written (the odd agent is copied).
template <int VEC>
__global__ void __launch_bounds__(kDefThreads)
    k_deffuant_step(const float *src, float *dst, int64_t n, int32_t B,
                    const int32_t *__restrict__ perm, const float *__restrict__ eps,
                    const float *__restrict__ mu) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = blockIdx.x * 64 + lane;
  if (q >= B / VEC) return;  // no barriers below
  const int col = q * VEC;
  float e[VEC], m[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    e[v] = eps[col + v];
    m[v] = mu[col + v];
  }
  const int64_t npairs = n >> 1;
  const int64_t stride = (int64_t)gridDim.y * kDefWaves;
  for (int64_t p0 = (int64_t)blockIdx.y * kDefWaves + wave; p0 < npairs;
       p0 += kDefStepPairs * stride) {
    // pairs p0, p0 + stride, ...; one past the end re-reads pair p0 and
    // stores nothing
    int64_t a[kDefStepPairs], c[kDefStepPairs];
    bool live[kDefStepPairs];
#pragma unroll
    for (int i = 0; i < kDefStepPairs; ++i) {
      const int64_t p = p0 + i * stride;
      live[i] = p < npairs;
      const int64_t pp = live[i] ? p : p0;
      a[i] = perm[2 * pp];
      c[i] = perm[2 * pp + 1];
    }
    float xa[kDefStepPairs][VEC], xc[kDefStepPairs][VEC];
#pragma unroll
    for (int i = 0; i < kDefStepPairs; ++i) {
      load_cols<VEC>(src + a[i] * B + col, xa[i]);
      load_cols<VEC>(src + c[i] * B + col, xc[i]);
    }
#pragma unroll
    for (int i = 0; i < kDefStepPairs; ++i) {
      float d[VEC], g[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) d[v] = xc[i][v] - xa[i][v];
      gates<VEC>([&](int v) { return e[v]; }, d, g);
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float delta = (m[v] * g[v]) * d[v];
        xa[i][v] = xa[i][v] + delta;
        xc[i][v] = xc[i][v] - delta;
      }
    }
#pragma unroll
    for (int i = 0; i < kDefStepPairs; ++i)
      if (live[i]) {
        store_cols<VEC>(dst + a[i] * B + col, xa[i]);
        store_cols<VEC>(dst + c[i] * B + col, xc[i]);
      }
  }
  if ((n & 1) && src != dst && blockIdx.y == 0 && wave == 0) {
    const int64_t r = perm[n - 1];
    float x[VEC];
    load_cols<VEC>(src + r * B + col, x);
    store_cols<VEC>(dst + r * B + col, x);
  }
}

// Pairs a wavefront holds in flight in the sweep: eight 1 KB row loads, as above.
// 65,536 x 256: 36.3 us a sweep against 37.3 with one pair and IEEE quotients, bound
// by the 192 MB that it moves.
constexpr int kDefSweepPairs = 2;

// Reverse sweep of one step: x_pre is the state before the step, lam holds
// dL/dx after it and is updated in place to dL/dx before it.
template <int VEC>
__global__ void __launch_bounds__(kDefThreads)
    k_deffuant_adjoint(const float *__restrict__ x_pre, float *__restrict__ lam, int64_t n,
                       int32_t B, const int32_t *__restrict__ perm,
                       const float *__restrict__ eps, const float *__restrict__ mu,
                       double *__restrict__ acc) {
  __shared__ double red[2][kDefWaves][64 * VEC];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = blockIdx.x * 64 + lane;
  const bool active = q < B / VEC;
  const int col = q * VEC;
  double ge[VEC], gm[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) ge[v] = gm[v] = 0.0;
  if (active) {
    float e[VEC], m[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      e[v] = eps[col + v];
      m[v] = mu[col + v];
    }
    const int64_t npairs = n >> 1;
    const int64_t stride = (int64_t)gridDim.y * kDefWaves;
    for (int64_t p0 = (int64_t)blockIdx.y * kDefWaves + wave; p0 < npairs;
         p0 += kDefSweepPairs * stride) {
      // pairs p0, p0 + stride; one past the end re-reads pair p0 and counts
      // and stores nothing
      int64_t a[kDefSweepPairs], c[kDefSweepPairs];
      bool live[kDefSweepPairs];
#pragma unroll
      for (int i = 0; i < kDefSweepPairs; ++i) {
        const int64_t p = p0 + i * stride;
        live[i] = p < npairs;
        const int64_t pp = live[i] ? p : p0;
        a[i] = perm[2 * pp];
        c[i] = perm[2 * pp + 1];
      }
      float xa[kDefSweepPairs][VEC], xc[kDefSweepPairs][VEC];
      float la[kDefSweepPairs][VEC], lc[kDefSweepPairs][VEC];
#pragma unroll
      for (int i = 0; i < kDefSweepPairs; ++i) {
        load_cols<VEC>(x_pre + a[i] * B + col, xa[i]);
        load_cols<VEC>(x_pre + c[i] * B + col, xc[i]);
        load_cols<VEC>(lam + a[i] * B + col, la[i]);
        load_cols<VEC>(lam + c[i] * B + col, lc[i]);
      }
#pragma unroll
      for (int i = 0; i < kDefSweepPairs; ++i) {
        float d[VEC], g[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v) d[v] = xc[i][v] - xa[i][v];
        gates<VEC>([&](int v) { return e[v]; }, d, g);
        if (!live[i]) continue;
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const float gp = div_gate_scale(g[v] * (1.0f - g[v]));
          const float fd = m[v] * (g[v] - fabsf(d[v]) * gp);
          const float fe = m[v] * d[v] * gp;
          const float fm = g[v] * d[v];
          const float w = la[i][v] - lc[i][v];
          la[i][v] = la[i][v] - w * fd;
          lc[i][v] = lc[i][v] + w * fd;
          ge[v] += (double)(w * fe);
          gm[v] += (double)(w * fm);
        }
        store_cols<VEC>(lam + a[i] * B + col, la[i]);
        store_cols<VEC>(lam + c[i] * B + col, lc[i]);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    red[0][wave][lane * VEC + v] = ge[v];
    red[1][wave][lane * VEC + v] = gm[v];
  }
  __syncthreads();
  if (wave == 0 && active) {
    double *slot = acc + (int64_t)blockIdx.y * 2 * B;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      double se = 0.0, sm = 0.0;
      for (int w = 0; w < kDefWaves; ++w) {
        se += red[0][w][lane * VEC + v];
        sm += red[1][w][lane * VEC + v];
      }
      slot[col + v] += se;
      slot[B + col + v] += sm;
    }
  }
}

// 1 / (1 + t) for t >= 0 in float64: the hardware reciprocal estimate
// (v_rcp_f64) refined by two Newton-Raphson steps r += r (1 - d r), a few
// FMAs instead of the IEEE division sequence; accurate to float64 rounding
// (a few ulps), far inside the statistics' 1e-10 tolerance.
__device__ __forceinline__ double inv_one_plus(double t) {
  const double d = 1.0 + t;
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  r = fma(r, fma(-d, r, 1.0), r);
  return r;
}

// Per-chunk float64 partial sums of the instance columns:
// [sum x, sum (x - 1/2)^2, hist_0 .. hist_31] -> partial[chunk][34][B].
// sigmoid(128 (x - k/32)) = 1 / (1 + t e^(4k)) with t = e^(-128 x).
// A workgroup is `cols` columns (a power of two, up to its threads) by
// kDefThreads / cols chunks, so that a small batch fills its lanes too.  What
// a chunk is and how the chunks are summed depends on n and the caller's number
// of chunks alone, not on the batch an instance runs in.  Bound by the 33
// reciprocals an opinion (float64 VALU).
__global__ void __launch_bounds__(kDefThreads)
    k_deffuant_stats(const float *__restrict__ x, int64_t n, int32_t B, int32_t cols,
                     int64_t rows, int64_t chunks, double *__restrict__ partial) {
  const int b = blockIdx.x * cols + (threadIdx.x & (cols - 1));
  const int64_t chunk = (int64_t)blockIdx.y * (kDefThreads / cols) + threadIdx.x / cols;
  if (b >= B || chunk >= chunks) return;
  const int64_t i0 = chunk * rows;
  const int64_t i1 = i0 + rows < n ? i0 + rows : n;
  const double e4 = exp(4.0);
  double s1 = 0.0, s2 = 0.0, h[kHistBins];
#pragma unroll
  for (int k = 0; k < kHistBins; ++k) h[k] = 0.0;
  for (int64_t i = i0; i < i1; ++i) {
    const double xi = (double)x[i * B + b];
    s1 += xi;
    s2 += (xi - 0.5) * (xi - 0.5);
    double t = exp(-kHistSlope * xi);
    double prev = inv_one_plus(t);
#pragma unroll
    for (int k = 0; k < kHistBins; ++k) {
      t *= e4;
      const double cur = inv_one_plus(t);
      h[k] += prev - cur;
      prev = cur;
    }
  }
  double *out = partial + chunk * kStatLen * B + b;
  out[0] = s1;
  out[B] = s2;
#pragma unroll
  for (int k = 0; k < kHistBins; ++k) out[(int64_t)(2 + k) * B] = h[k];
}

// out[j][b] = sum over r of in[r][j][b], for j = blockIdx.y; 64 columns per
// block, kSumGroups row groups of four loads in flight, combined in a fixed
// order.  Few rows have fewer groups, a wavefront each (an empty one adds nothing,
// and 100,000 instances of one row took 105 us with 16 each, 21 with 4).
constexpr int kSumGroups = 16;

__global__ void __launch_bounds__(64 * kSumGroups)
    k_sum_rows(const double *__restrict__ in, int64_t rows, int32_t J, int32_t B,
               double *__restrict__ out) {
  __shared__ double red[kSumGroups][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int b = blockIdx.x * 64 + lane;
  const int j = blockIdx.y;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  if (b < B) {
    for (int64_t r = g; r < rows; r += 4 * kSumGroups) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[u] = r + u * kSumGroups < rows ? in[((r + u * kSumGroups) * J + j) * B + b] : 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] += v[u];
    }
  }
  red[g][lane] = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  if (g == 0 && b < B) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += red[q][lane];
    out[(int64_t)j * B + b] = t;
  }
}

// stats[b][34], loss[b] and the coefficients of dL/dx (coef[34][B]:
// dL/dmean / n, dL/dvar * 2 / n, dL/dhist_k / n) from the column sums.
// weights (optional, [34]): L = sum_j w_j (stats_j - target_j)^2.
__global__ void k_deffuant_loss(const double *__restrict__ sums, int64_t n, int32_t B,
                                const double *__restrict__ target,
                                const double *__restrict__ weights, double *__restrict__ stats,
                                double *__restrict__ loss, double *__restrict__ coef) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const double dn = (double)n;
  double sum[kStatLen], aim[kStatLen], wt[kStatLen];  // all loads in flight at once
#pragma unroll
  for (int k = 0; k < kStatLen; ++k) {
    sum[k] = sums[(int64_t)k * B + b];
    aim[k] = target[k];
    wt[k] = weights ? weights[k] : 1.0;
  }
  const double m = sum[0] / dn;
  const double v = sum[1] / dn - (m - 0.5) * (m - 0.5);
  const double w0 = wt[0], w1 = wt[1];
  double L = w0 * (m - aim[0]) * (m - aim[0]) + w1 * (v - aim[1]) * (v - aim[1]);
  stats[(int64_t)b * kStatLen] = m;
  stats[(int64_t)b * kStatLen + 1] = v;
  coef[b] = w0 * 2.0 * (m - aim[0]) / dn;
  coef[B + b] = w1 * 2.0 * (v - aim[1]) * 2.0 / dn;
#pragma unroll
  for (int k = 0; k < kHistBins; ++k) {
    const double hk = sum[2 + k] / dn;
    const double wk = wt[2 + k];
    stats[(int64_t)b * kStatLen + 2 + k] = hk;
    L += wk * (hk - aim[2 + k]) * (hk - aim[2 + k]);
    coef[(int64_t)(2 + k) * B + b] = wk * 2.0 * (hk - aim[2 + k]) / dn;
  }
  loss[b] = L;
}

// dL/dx for the final opinion x of an agent of instance b.
__device__ __forceinline__ float lambda_at(float x, int b, int32_t B,
                                           const double *__restrict__ stats,
                                           const double *__restrict__ coef) {
  const double xi = (double)x;
  const double e4 = exp(4.0);
  double g = coef[b] + coef[B + b] * (xi - stats[(int64_t)b * kStatLen]);
  double t = exp(-kHistSlope * xi);
  double s = inv_one_plus(t);
  double ds_prev = s * (1.0 - s);
  for (int k = 0; k < kHistBins; ++k) {
    t *= e4;
    s = inv_one_plus(t);
    const double ds = s * (1.0 - s);
    g += coef[(int64_t)(2 + k) * B + b] * kHistSlope * (ds_prev - ds);
    ds_prev = ds;
  }
  return (float)g;
}

// lam[i][b] = dL/dx_i for instance b from the final state.
__global__ void k_deffuant_lambda(const float *__restrict__ x, int64_t n, int32_t B,
                                  const double *__restrict__ stats,
                                  const double *__restrict__ coef, float *__restrict__ lam) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * B) return;
  lam[idx] = lambda_at(x[idx], (int)(idx % B), B, stats, coef);
}

// ---- column runs: one workgroup, one instance, all steps in one launch
//
// The opinions x (and in the backward the adjoints lam) of one instance live
// in LDS, indexed by agent; a step is, per pair, two LDS reads, the gate, two
// LDS writes, and one barrier.  HBM sees the pairings (shared by all
// instances, so mostly L2), the checkpoints, and a tape of the pairs'
// differences d = x_c - x_a: a step's adjoint needs nothing else of the
// state, and in pair order the tape is written and read coalesced, at 2 bytes
// an agent and step where a step kernel moves 8 (forward) or 12 (adjoint).
// What bounds a step is then the gate's arithmetic (VALU).
//
// Layouts: ckpt[0] and work as ever ([n][B]); ckpt[j], j >= 1, and lam as
// [B][n]; tape of one step [B][n / 2], a segment's steps in traj (k n / 2 <=
// (k - 1) n floats an instance for k >= 2).  With k = 1 there are no
// checkpoints to recompute from: step t's tape takes the first half of
// ckpt[t] (step 0's the second half of ckpt[1]), and every backward sweeps it.
constexpr int kColLds = 160 * 1024;
constexpr int kColStatic = 512;                          // reduction scratch
constexpr int64_t kColAgents = (kColLds - kColStatic) / 4;  // n floats in LDS
constexpr int kColThreads = 1024;
// P, the pairs a thread holds per iteration: 1 while a thread has no more than
// one pair (a step is then one chain of latencies), 4 where it has several.

struct ColumnRun {
  int32_t n, B, steps, k;
  const int32_t *perms;
  const float *eps, *mu;
  float *work, *ckpt, *traj, *lam;
  double *grads;
  int32_t tape_last;  // traj holds (forward: receives) the last segment's tape
};

// Instance of workgroup blk.  Workgroups go to the 8 XCDs in turn; within 256
// of them each XCD gets 32 neighbouring instances, one 128-byte line of a row
// of [n][B], so that its L2 reads and writes those rows whole.
__device__ __forceinline__ int32_t column_of(int32_t blk, int32_t B) {
  const int32_t base = blk & ~255, r = blk & 255;
  return base + 256 <= B ? base + (r & 7) * 32 + (r >> 3) : blk;
}

// Accesses below go through raw buffers of one row: a pair past the end loads
// pair (0, 0) and stores nothing, without a branch around the access (which
// would make every later wait a full one).
using ColBuffer = __amdgpu_buffer_rsrc_t;
using ColPair = unsigned __attribute__((ext_vector_type(2)));
__device__ __forceinline__ ColBuffer col_buffer(const void *p, int32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000);
}

// Threads of the workgroup: with P > 1 always kColThreads.
template <int P>
__device__ __forceinline__ int32_t col_threads() {
  return P > 1 ? kColThreads : (int32_t)__builtin_amdgcn_readfirstlane(blockDim.x);
}

// A step's pairs in rounds of P x kColThreads (P = 1: one round).
template <int P>
__device__ __forceinline__ int32_t col_rounds(int32_t npairs) {
  return P > 1 ? (npairs + P * kColThreads - 1) / (P * kColThreads) : 1;
}

// Pair u of a thread in round r.
template <int P>
__device__ __forceinline__ int32_t col_pair(int32_t r, int u) {
  return (r * P + u) * kColThreads + (int32_t)threadIdx.x;
}

template <int P>
struct ColPairs {
  ColPair p[P];
};
template <int P>
__device__ __forceinline__ ColPairs<P> load_pairs(const ColumnRun &a, int32_t t, int32_t r) {
  ColPairs<P> v;
  const ColBuffer b = col_buffer(a.perms + (int64_t)t * a.n, 8 * (a.n >> 1));
#pragma unroll
  for (int u = 0; u < P; ++u)
    v.p[u] = __builtin_amdgcn_raw_buffer_load_b64(b, 8 * col_pair<P>(r, u), 0, 0);
  return v;
}

// Steps t0 .. t1 - 1 on the opinions x; step t's differences go to tape(t)
// where that is not null; after(t) runs with every thread past step t.
template <int P, class Tape, class After>
__device__ __forceinline__ void column_steps(const ColumnRun &a, float *x, int32_t t0, int32_t t1,
                                             float eps, float mu, Tape tape, After after) {
  const int32_t npairs = a.n >> 1, rounds = col_rounds<P>(npairs);
  ColPairs<P> pr = load_pairs<P>(a, t0, 0);
  for (int32_t t = t0; t < t1; ++t) {
    float *out = tape(t);
    const ColBuffer tb = col_buffer(out, out ? 4 * npairs : 0);
    for (int32_t r = 0; r < rounds; ++r) {
      // the next pairs, of this step or the next (after the last: its own)
      const bool more = r + 1 < rounds;
      const ColPairs<P> nx =
          load_pairs<P>(a, more || t + 1 == t1 ? t : t + 1, more ? r + 1 : 0);
      float xa[P], xc[P], d[P], g[P];
#pragma unroll
      for (int u = 0; u < P; ++u) {
        xa[u] = x[pr.p[u].x];
        xc[u] = x[pr.p[u].y];
        d[u] = xc[u] - xa[u];
      }
      gates<P>([eps](int) { return eps; }, d, g);
#pragma unroll
      for (int u = 0; u < P; ++u) {
        const float delta = (mu * g[u]) * d[u];
        if (col_pair<P>(r, u) < npairs) {
          x[pr.p[u].x] = xa[u] + delta;
          x[pr.p[u].y] = xc[u] - delta;
        }
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(d[u]), tb, 4 * col_pair<P>(r, u), 0,
                                              0);
      }
      pr = nx;
    }
    lds_barrier();
    after(t);
  }
}

// Row of step t's tape in the k = 1 layout.
__device__ __forceinline__ float *column_full_tape(const ColumnRun &a, int32_t t, int32_t b) {
  const int64_t nB = (int64_t)a.n * a.B, half = a.n >> 1;
  return a.ckpt + (t ? t * nB : nB + half * a.B) + half * b;
}

template <int P>
__global__ void __launch_bounds__(kColThreads) k_deffuant_column_forward(ColumnRun a) {
  extern __shared__ float col_x[];
  const int32_t b = column_of(blockIdx.x, a.B), tid = threadIdx.x, T = col_threads<P>();
  const int64_t nB = (int64_t)a.n * a.B, half = a.n >> 1;
  for (int32_t i = tid; i < a.n; i += T) col_x[i] = a.ckpt[(int64_t)i * a.B + b];
  lds_barrier();
  const int32_t t_last = (a.steps - 1) / a.k * a.k;
  int32_t next = a.k;  // steps done at the next checkpoint
  auto tape = [&](int32_t t) -> float * {
    if (a.k == 1) return column_full_tape(a, t, b);
    return a.tape_last && t >= t_last ? a.traj + (t - t_last) * half * a.B + half * b : nullptr;
  };
  auto after = [&](int32_t t) {
    if (a.k == 1 || t + 1 != next || t + 1 == a.steps) return;
    float *c = a.ckpt + (int64_t)((t + 1) / a.k) * nB + (int64_t)b * a.n;
    for (int32_t i = tid; i < a.n; i += T) c[i] = col_x[i];
    next += a.k;
    lds_barrier();  // before the next step writes
  };
  column_steps<P>(a, col_x, 0, a.steps, a.eps[b], a.mu[b], tape, after);
  for (int32_t i = tid; i < a.n; i += T) a.work[(int64_t)i * a.B + b] = col_x[i];
}

// Reverse sweep of steps t1 - 1 .. t0 on the adjoints l.
template <int P, class Tape>
__device__ __forceinline__ void column_sweep(const ColumnRun &a, float *l, int32_t t0, int32_t t1,
                                             float eps, float mu, Tape tape, double &ge,
                                             double &gm) {
  const int32_t npairs = a.n >> 1, rounds = col_rounds<P>(npairs);
  auto load_d = [&](int32_t t, int32_t r, float (&d)[P]) {
    const ColBuffer tb = col_buffer(tape(t), 4 * npairs);
#pragma unroll
    for (int u = 0; u < P; ++u)
      d[u] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(tb, 4 * col_pair<P>(r, u), 0, 0));
  };
  ColPairs<P> pr = load_pairs<P>(a, t1 - 1, 0);
  float d[P];
  load_d(t1 - 1, 0, d);
  for (int32_t t = t1 - 1; t >= t0; --t) {
    for (int32_t r = 0; r < rounds; ++r) {
      const bool more = r + 1 < rounds;
      const int32_t tn = more || t == t0 ? t : t - 1, rn = more ? r + 1 : 0;
      const ColPairs<P> nx = load_pairs<P>(a, tn, rn);
      float dn[P], la[P], lc[P], g[P];
      load_d(tn, rn, dn);
#pragma unroll
      for (int u = 0; u < P; ++u) {
        la[u] = l[pr.p[u].x];
        lc[u] = l[pr.p[u].y];
      }
      gates<P>([eps](int) { return eps; }, d, g);
#pragma unroll
      for (int u = 0; u < P; ++u) {
        const float gp = div_gate_scale(g[u] * (1.0f - g[u]));
        const float fd = mu * (g[u] - fabsf(d[u]) * gp);
        const float fe = mu * d[u] * gp;
        const float fm = g[u] * d[u];
        const bool pair = col_pair<P>(r, u) < npairs;
        const float w = pair ? la[u] - lc[u] : 0.0f;
        if (pair) {
          l[pr.p[u].x] = la[u] - w * fd;
          l[pr.p[u].y] = lc[u] + w * fd;
        }
        ge += (double)(w * fe);
        gm += (double)(w * fm);
        d[u] = dn[u];
      }
      pr = nx;
    }
    lds_barrier();
  }
}

// The whole backward of one instance: per segment from the last, the steps
// again from its checkpoint with their tape (unless the forward left it),
// then the sweep.  kBoth: x and lam both fit LDS; otherwise they take turns,
// lam waiting in its global column meanwhile.
template <bool kBoth, int P>
__global__ void __launch_bounds__(kColThreads) k_deffuant_column_backward(ColumnRun a) {
  extern __shared__ float col_mem[];
  __shared__ double red[2][kColThreads / 64];
  const int32_t b = column_of(blockIdx.x, a.B), tid = threadIdx.x, T = col_threads<P>();
  const int64_t nB = (int64_t)a.n * a.B, half = a.n >> 1;
  float *x = col_mem, *l = kBoth ? col_mem + a.n : col_mem;
  float *column = a.lam + (int64_t)b * a.n;
  const float eps = a.eps[b], mu = a.mu[b];
  double ge = 0.0, gm = 0.0;
  const int32_t len = a.k == 1 ? a.steps : a.k;  // steps a segment
  const int32_t nseg = (a.steps + len - 1) / len;
  for (int32_t j = nseg - 1; j >= 0; --j) {
    const int32_t t0 = j * len, t1 = t0 + len < a.steps ? t0 + len : a.steps;
    auto tape = [&](int32_t t) -> float * {
      return a.k == 1 ? column_full_tape(a, t, b) : a.traj + (t - t0) * half * a.B + half * b;
    };
    if (a.k > 1 && !(a.tape_last && j == nseg - 1)) {
      if (j == 0) {
        for (int32_t i = tid; i < a.n; i += T) x[i] = a.ckpt[(int64_t)i * a.B + b];
      } else {
        const float *c = a.ckpt + j * nB + (int64_t)b * a.n;
        for (int32_t i = tid; i < a.n; i += T) x[i] = c[i];
      }
      lds_barrier();
      column_steps<P>(a, x, t0, t1, eps, mu, tape, [](int32_t) {});
    }
    if (!kBoth || j == nseg - 1) {
      for (int32_t i = tid; i < a.n; i += T) l[i] = column[i];
      lds_barrier();
    }
    column_sweep<P>(a, l, t0, t1, eps, mu, tape, ge, gm);
    if (!kBoth && j > 0) {
      for (int32_t i = tid; i < a.n; i += T) column[i] = l[i];
      __syncthreads();
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    ge += __shfl_xor(ge, off);
    gm += __shfl_xor(gm, off);
  }
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = ge;
    red[1][tid >> 6] = gm;
  }
  __syncthreads();
  if (tid < 2) {
    double s = 0.0;
    for (int w = 0; w < (T >> 6); ++w) s += red[tid][w];
    a.grads[(int64_t)tid * a.B + b] = s;
  }
}

// k_deffuant_lambda into columns: lam[b][i], tiles of R agents x 16 instances
// turned in LDS; R = 64 writes whole lines, R = 16 spreads a small batch over
// more workgroups (1,001 x 12: 18 us with 64, 8 with 16).
template <int R>
__global__ void __launch_bounds__(256)
    k_deffuant_lambda_columns(const float *__restrict__ x, int64_t n, int32_t B,
                              const double *__restrict__ stats, const double *__restrict__ coef,
                              float *__restrict__ lam) {
  __shared__ float tile[16][R + 1];
  const int64_t i0 = (int64_t)blockIdx.x * R;
  const int32_t b0 = blockIdx.y * 16;
#pragma unroll 1
  for (int r = threadIdx.x >> 4; r < R; r += 16) {
    const int c = threadIdx.x & 15;
    const int64_t i = i0 + r;
    if (i < n && b0 + c < B) tile[c][r] = lambda_at(x[i * B + b0 + c], b0 + c, B, stats, coef);
  }
  __syncthreads();
  for (int c = threadIdx.x / R; c < 16; c += 256 / R) {
    const int r = threadIdx.x & (R - 1);
    if (i0 + r < n && b0 + c < B) lam[(int64_t)(b0 + c) * n + i0 + r] = tile[c][r];
  }
}

__global__ void k_deffuant_init(const uint32_t *__restrict__ init_key, int64_t n, int32_t B,
                                float *__restrict__ x, int mode) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float v = unit_float(bits_scalar(split_at(Key{init_key[0], init_key[1]}, n, i, mode), mode));
  for (int32_t b = 0; b < B; ++b) x[i * B + b] = v;
}

__global__ void k_fill_f64(double *__restrict__ p, int64_t n, double v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// VEC = 4 when every row segment is 16-byte aligned.
inline bool use_vec4(int32_t B, const void *a, const void *b) {
  return (B % 4) == 0 && aligned16(a) && aligned16(b);
}

void launch_step(const float *src, float *dst, int64_t n, int32_t B, const int32_t *perm,
                 const float *eps, const float *mu, int32_t pair_blocks, hipStream_t s) {
  if (use_vec4(B, src, dst)) {
    const dim3 g(nblocks(B / 4, 64), (unsigned)pair_blocks);
    hipLaunchKernelGGL(k_deffuant_step<4>, g, dim3(kDefThreads), 0, s, src, dst, n, B, perm,
                       eps, mu);
  } else {
    const dim3 g(nblocks(B, 64), (unsigned)pair_blocks);
    hipLaunchKernelGGL(k_deffuant_step<1>, g, dim3(kDefThreads), 0, s, src, dst, n, B, perm,
                       eps, mu);
  }
}

void launch_adjoint(const float *x_pre, float *lam, int64_t n, int32_t B, const int32_t *perm,
                    const float *eps, const float *mu, int32_t pair_blocks, double *acc,
                    hipStream_t s) {
  if (use_vec4(B, x_pre, lam)) {
    const dim3 g(nblocks(B / 4, 64), (unsigned)pair_blocks);
    hipLaunchKernelGGL(k_deffuant_adjoint<4>, g, dim3(kDefThreads), 0, s, x_pre, lam, n, B,
                       perm, eps, mu, acc);
  } else {
    const dim3 g(nblocks(B, 64), (unsigned)pair_blocks);
    hipLaunchKernelGGL(k_deffuant_adjoint<1>, g, dim3(kDefThreads), 0, s, x_pre, lam, n, B,
                       perm, eps, mu, acc);
  }
}

void launch_sum_rows(const double *in, int64_t rows, int32_t J, int32_t B, double *out,
                     hipStream_t s) {
  const unsigned groups = rows < kSumGroups ? (unsigned)rows : (unsigned)kSumGroups;
  hipLaunchKernelGGL(k_sum_rows, dim3(nblocks(B, 64), (unsigned)J), dim3(64 * groups), 0, s, in,
                     rows, J, B, out);
}

void launch_loss(const abm_deffuant_problem *p, const float *x, hipStream_t s) {
  int32_t cols = 1;
  while (cols < p->batch && cols < kDefThreads) cols *= 2;
  const int64_t most = p->stat_chunks < kStatChunks ? p->stat_chunks : kStatChunks;
  const int64_t rows = (p->n + most - 1) / most;
  const int64_t chunks = (p->n + rows - 1) / rows;
  hipLaunchKernelGGL(k_deffuant_stats,
                     dim3(nblocks(p->batch, cols), nblocks(chunks, kDefThreads / cols)),
                     dim3(kDefThreads), 0, s, x, p->n, p->batch, cols, rows, chunks, p->partial);
  launch_sum_rows(p->partial, chunks, kStatLen, p->batch, p->sums, s);
  hipLaunchKernelGGL(k_deffuant_loss, dim3(nblocks(p->batch, 64)), dim3(64), 0, s,
                     (const double *)p->sums, p->n, p->batch, p->target, p->weights, p->stats,
                     p->loss, p->coef);
}

// Above so many agents (three rounds of pairs a step) a column costs more than
// the step kernels do for a few instances: forward and backward of 60 steps, 1
// instance of 34,000 agents, 1,303 us in columns and 865 in step kernels; 9 of
// 30,000, 1,102 and 985; 17 of 30,000, 1,140 and 1,056, but 3,254 and 3,414 with
// 200 steps.  With 24,576 agents, 1 instance 872 and 840, 17 instances 902 and
// 982.  A multiple of four instances takes four a lane in the step kernels, and
// as long as 64: 4 of 40,000, 1,366 and 2,567.
constexpr int64_t kColFewAgents = 3 * 2 * 4 * kColThreads;
constexpr int32_t kColFewInstances = 16;
// Populations of up to four pairs leave a column's lanes idle, which tells once
// the instances fill the chip seven times over (8,192 wavefronts): 64,000 instances
// of 8 agents, 60 steps, 914 us in columns and 811 in step kernels, of 2 agents 884
// and 669, of 32 agents 963 and 1,719; 32,000 of 8, 538 and 835.
constexpr int64_t kColPairAgents = 8;
constexpr int32_t kColManyInstances = 7 * 8192;

// Whether a flagged descriptor takes the column run; the same answer in the
// forward and the backward of one descriptor.  Either way the same opinions,
// statistics and terms of the gradients, those summed in another order.
bool column_run(const abm_deffuant_problem *p) {
  if (!(p->flags & ABM_DEFFUANT_COLUMNS) || p->n > kColAgents || p->steps < 1) return false;
  if (p->ckpt_every == 1 ? p->steps < 2 : !p->traj) return false;
  if (p->n > kColFewAgents && p->batch <= kColFewInstances && p->batch % 4 != 0) return false;
  return p->n > kColPairAgents || p->batch <= kColManyInstances;
}

ColumnRun column_args(const abm_deffuant_problem *p) {
  ColumnRun a;
  a.n = (int32_t)p->n;
  a.B = p->batch;
  a.steps = p->steps;
  a.k = p->ckpt_every;
  a.perms = p->perms;
  a.eps = p->eps;
  a.mu = p->mu;
  a.work = p->work;
  a.ckpt = p->ckpt;
  a.traj = p->traj;
  a.lam = p->lam;
  a.grads = p->grads;
  a.tape_last = (p->flags & ABM_DEFFUANT_TAPE_LAST) != 0;
  return a;
}

// One pair a thread, whole wavefronts, up to a full workgroup.
unsigned column_threads(int64_t n) {
  const int64_t t = ((n >> 1) + 63) / 64 * 64;
  return (unsigned)(t < kColThreads ? t : kColThreads);
}

using ColumnKernel = void (*)(ColumnRun);

ColumnKernel column_forward(int64_t n) {
  return (n >> 1) <= kColThreads ? k_deffuant_column_forward<1> : k_deffuant_column_forward<4>;
}

bool column_both(int64_t n) { return 2 * n <= kColAgents; }

ColumnKernel column_backward(int64_t n) {
  if ((n >> 1) <= kColThreads) return k_deffuant_column_backward<true, 1>;
  return column_both(n) ? k_deffuant_column_backward<true, 4>
                        : k_deffuant_column_backward<false, 4>;
}

constexpr int kMaxDevices = 64;
std::mutex g_column_attr_mu;
bool g_column_attr_set[kMaxDevices];

// The column kernels need more than 64 KB of dynamic LDS: the limit is raised
// once per device, under a lock.
int column_lds_attr() {
  int dev = -1;
  ABM_CHECK_HIP(hipGetDevice(&dev));
  ABM_REQUIRE(dev >= 0 && dev < kMaxDevices, "deffuant: device index out of range");
  std::lock_guard<std::mutex> lock(g_column_attr_mu);
  if (!g_column_attr_set[dev]) {
    for (const ColumnKernel k :
         {k_deffuant_column_forward<1>, k_deffuant_column_forward<4>,
          k_deffuant_column_backward<true, 1>, k_deffuant_column_backward<true, 4>,
          k_deffuant_column_backward<false, 4>})
      ABM_CHECK_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)(kColAgents * 4)));
    g_column_attr_set[dev] = true;
  }
  return kOk;
}

int check_problem(const abm_deffuant_problem *p, const char *who, bool backward) {
  bool ok = p && p->n >= 2 && p->n < (1ll << 31) && p->batch >= 1 && p->steps >= 0 &&
            p->ckpt_every >= 1 && p->pair_blocks >= 1 && p->pair_blocks <= 65535 &&
            p->stat_chunks >= 1 && p->stat_chunks <= 65535 && p->n * (int64_t)p->batch < (1ll << 40) &&
            p->perms && p->eps && p->mu && p->work && p->ckpt && p->partial && p->sums &&
            p->coef && p->target && p->stats && p->loss;
  if (ok && backward)
    ok = p->lam && p->acc && p->grads && (p->ckpt_every == 1 || p->traj);
  if (!ok) {
    set_error(std::string(who) + ": bad problem descriptor");
    return kErrInvalid;
  }
  return kOk;
}

}  // namespace abm

using namespace abm;

extern "C" {

int abm_deffuant_init(const uint32_t *init_key, int64_t n, int32_t batch, float *x, int mode,
                      void *stream) {
  ABM_REQUIRE(init_key && x && n >= 1 && n < (1ll << 31) && batch >= 1 &&
                  (mode == 0 || mode == 1),
              "abm_deffuant_init: bad arguments");
  hipLaunchKernelGGL(k_deffuant_init, dim3(nblocks(n, 256)), dim3(256), 0, (hipStream_t)stream,
                     init_key, n, batch, x, mode);
  ABM_LAUNCH_CHECK("abm_deffuant_init");
  return kOk;
}

int abm_deffuant_step(const float *src, float *dst, int64_t n, int32_t batch,
                      const int32_t *perm, const float *eps, const float *mu,
                      int32_t pair_blocks, void *stream) {
  ABM_REQUIRE(src && dst && perm && eps && mu && n >= 1 && n < (1ll << 31) && batch >= 1 &&
                  pair_blocks >= 1 && pair_blocks <= 65535,
              "abm_deffuant_step: bad arguments");
  launch_step(src, dst, n, batch, perm, eps, mu, pair_blocks, (hipStream_t)stream);
  ABM_LAUNCH_CHECK("abm_deffuant_step");
  return kOk;
}

int abm_deffuant_forward(const abm_deffuant_problem *p, void *stream) {
  if (int rc = check_problem(p, "abm_deffuant_forward", false)) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (column_run(p)) {
    if (int rc = column_lds_attr()) return rc;
    hipLaunchKernelGGL(column_forward(p->n), dim3((unsigned)p->batch),
                       dim3(column_threads(p->n)), (size_t)p->n * 4, s, column_args(p));
    launch_loss(p, p->work, s);
    ABM_LAUNCH_CHECK("abm_deffuant_forward");
    return kOk;
  }
  const int64_t nB = p->n * (int64_t)p->batch;
  const int32_t k = p->ckpt_every;
  // first step of the last segment; with the tape flag its steps write traj
  // out of place (the backward then skips recomputing it)
  const int32_t t_last = p->steps > 0 ? (p->steps - 1) / k * k : 0;
  const bool tape = (p->flags & ABM_DEFFUANT_TAPE_LAST) && p->traj && k > 1;
  const float *src = p->ckpt;
  for (int32_t t = 0; t < p->steps; ++t) {
    const bool to_ckpt = ((t + 1) % k) == 0 && t + 1 < p->steps;
    float *dst = p->work;
    if (to_ckpt)
      dst = p->ckpt + (int64_t)((t + 1) / k) * nB;
    else if (tape && t >= t_last && t + 1 < p->steps)
      dst = p->traj + (int64_t)(t - t_last) * nB;
    launch_step(src, dst, p->n, p->batch, p->perms + (int64_t)t * p->n, p->eps, p->mu,
                p->pair_blocks, s);
    src = dst;
  }
  launch_loss(p, p->steps > 0 ? p->work : p->ckpt, s);
  ABM_LAUNCH_CHECK("abm_deffuant_forward");
  return kOk;
}

int abm_deffuant_backward(const abm_deffuant_problem *p, void *stream) {
  if (int rc = check_problem(p, "abm_deffuant_backward", true)) return rc;
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = p->n, nB = n * (int64_t)p->batch;
  const int32_t k = p->ckpt_every;
  const float *final_x = p->steps > 0 ? p->work : p->ckpt;
  if (column_run(p)) {
    if (int rc = column_lds_attr()) return rc;
    const bool wide = nblocks(n, 64) * (int64_t)nblocks(p->batch, 16) >= 1024;
    hipLaunchKernelGGL(wide ? k_deffuant_lambda_columns<64> : k_deffuant_lambda_columns<16>,
                       dim3(nblocks(n, wide ? 64 : 16), nblocks(p->batch, 16)), dim3(256), 0, s,
                       final_x, n, p->batch, (const double *)p->stats, (const double *)p->coef,
                       p->lam);
    hipLaunchKernelGGL(column_backward(n), dim3((unsigned)p->batch), dim3(column_threads(n)),
                       (size_t)n * (column_both(n) ? 8 : 4), s, column_args(p));
    ABM_LAUNCH_CHECK("abm_deffuant_backward");
    return kOk;
  }
  hipLaunchKernelGGL(k_deffuant_lambda, dim3(nblocks(nB, 256)), dim3(256), 0, s, final_x, n,
                     p->batch, (const double *)p->stats, (const double *)p->coef, p->lam);
  const int64_t acc_len = (int64_t)p->pair_blocks * 2 * p->batch;
  hipLaunchKernelGGL(k_fill_f64, dim3(nblocks(acc_len, 256)), dim3(256), 0, s, p->acc, acc_len,
                     0.0);
  const int32_t nseg = (p->steps + k - 1) / k;
  for (int32_t j = nseg - 1; j >= 0; --j) {
    const int32_t t0 = j * k, t1 = t0 + k < p->steps ? t0 + k : p->steps;
    const float *ck = p->ckpt + (int64_t)j * nB;
    const float *src = ck;
    const bool taped = j == nseg - 1 && (p->flags & ABM_DEFFUANT_TAPE_LAST);
    for (int32_t u = 0; !taped && u + 1 < t1 - t0; ++u) {
      float *dst = p->traj + (int64_t)u * nB;
      launch_step(src, dst, n, p->batch, p->perms + (int64_t)(t0 + u) * n, p->eps, p->mu,
                  p->pair_blocks, s);
      src = dst;
    }
    for (int32_t t = t1 - 1; t >= t0; --t) {
      const float *pre = t == t0 ? ck : p->traj + (int64_t)(t - t0 - 1) * nB;
      launch_adjoint(pre, p->lam, n, p->batch, p->perms + (int64_t)t * n, p->eps, p->mu,
                     p->pair_blocks, p->acc, s);
    }
  }
  launch_sum_rows(p->acc, p->pair_blocks, 2, p->batch, p->grads, s);
  ABM_LAUNCH_CHECK("abm_deffuant_backward");
  return kOk;
}

}  // extern "C"
