// deffuant_gate.hpp -- the Deffuant gate 1 / (1 + exp(-(eps - |d|) / 0.02)) in
// float32, each operation rounded once, and a short form of it with the same
// bits.  Also for host code.
#pragma once

#include <cmath>

#include "abm_math.h"

namespace abm {

constexpr float kGateScale = 0.02f;

ABM_MATH_FN float gate(float eps, float d) {
  const float z = (eps - fabsf(d)) / kGateScale;
  const float e = abm_expf(-z);
  const float den = 1.0f + e;
  return 1.0f / den;
}

// x / kGateScale in three operations: with y = 50 the rounded reciprocal,
// q + (x - q c) y corrects q = x y to the rounded quotient (Markstein, IBM J. Res.
// Dev. 34(1), 1990).  Equal to the IEEE division for every float32 of 2^-105 <=
// |x| <= 1.6; below, where the remainder is rounded, it may be the float32 next
// to it.  A gate is 1 / 2 for all of those.  A sweep divides g (1 - g), which is
// 2^-87 or more for a gate of the short form; below 2^-105, of a gate() of |z|
// above 72, an ulp of that quotient is below 1e-36.
ABM_MATH_FN float div_gate_scale(float x) {
  const float q = x * 50.0f;
  return fmaf(fmaf(-q, kGateScale, x), 50.0f, q);
}

// 1 / d rounded once for 1 <= d < 2^120 from an estimate within 1 ulp of the
// rounded one, by two corrections (the second exact, Markstein as above).  Where
// every mantissa bit of d is set the estimate has to be the rounded one, as
// gfx950's v_rcp_f32 is: from 2^-k in its place 2^-k would come back.
ABM_MATH_FN float inv_rounded(float d, float estimate) {
  const float r = fmaf(fmaf(-d, estimate, 1.0f), estimate, estimate);
  return fmaf(fmaf(-d, r, 1.0f), r, r);
}

// gate() of num = eps - |d| for |num| <= kGateShort (|z| <= 60): its quotients as
// above, and abm_expf without its range branches.  rcp(d): the estimate of 1 / d.
constexpr float kGateShort = 1.2f;

template <class Rcp>
ABM_MATH_FN float gate_short(float num, Rcp rcp) {
  const float x = -div_gate_scale(num);
  const float m = __builtin_rintf(x * 0x1.715476p0f);
  const float r = (x - m * 0x1.62e4p-1f) - m * 0x1.7f7d1cp-20f;
  float q = 0x1.a01a02p-13f;
  q = 0x1.6c16c2p-10f + q * r;
  q = 0x1.111112p-7f + q * r;
  q = 0x1.555556p-5f + q * r;
  q = 0x1.555556p-3f + q * r;
  q = 0.5f + q * r;
  const float p = 1.0f + (r + (r * r) * q);
  const float d = 1.0f + __builtin_ldexpf(p, (int)m);  // exact: no subnormal here
  return inv_rounded(d, rcp(d));
}

}  // namespace abm
