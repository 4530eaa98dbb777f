// sin(x) and cos(x) of a positional-encoding argument, |x| <= kPeSincosMax, for
// the forms that round both to 16 bits.
//
// x minus the nearest multiple n of pi/2, pi/2 in two parts (Cody-Waite; the
// third would move x by 9e-12): the first fma is exact, the second's rounding
// error is kept in lo.  Then odd / even polynomials on [-0.79, 0.79] (minimax by
// iterated weighted least squares, 1.9e-9 and 1.0e-10 off; |r| passes pi/4 by at
// most 4e-4, where the rounded quotient picks the other neighbour).
// Against 64-bit values over |x| <= 512 and 8192: rms 1.5e-8, largest error
// 6.4e-8 for both (the library's 1.8e-8 and 7.0e-8; correctly rounded 1.5e-8 and
// 3.0e-8).  Without lo rms 1.7e-8.
//
// Plain C++ apart from the qualifiers, so that a host build can check the above.
#pragma once

#ifndef SAILOR_PE_FN
#define SAILOR_PE_FN __device__ __forceinline__
#endif

namespace sailor {

constexpr float kPeSincosMax = 8192.0f;

SAILOR_PE_FN void pe_sincos(float x, float& s, float& c) {
  const float n = __builtin_rintf(x * 0.63661977f);
  const float r1 = __builtin_fmaf(-n, 1.57079637f, x);
  const float r = __builtin_fmaf(-n, -4.37113883e-8f, r1);
  const float lo = __builtin_fmaf(-n, -4.37113883e-8f, r1 - r);
  const float z = r * r;
  float p = __builtin_fmaf(-1.9491608e-4f, z, 8.33194703e-3f);
  p = __builtin_fmaf(p, z, -1.66666508e-1f);
  float q = __builtin_fmaf(2.44342136e-5f, z, -1.38873316e-3f);
  q = __builtin_fmaf(q, z, 4.16666456e-2f);
  q = __builtin_fmaf(q, z, -0.5f);
  const float sr = r + __builtin_fmaf(p, z * r, lo);
  const float cr = __builtin_fmaf(q, __builtin_fmaf(lo + lo, r, z), 1.0f);
  const int m = (int)n;
  s = m & 1 ? cr : sr;
  c = m & 1 ? sr : cr;
  s = m & 2 ? -s : s;
  c = (m + 1) & 2 ? -c : c;
}

}  // namespace sailor
