// abl_root_rcp.hpp -- the rounding steps of the correctly rounded single-precision
// root and reciprocal of abl_device.hpp, from the approximations that the
// instructions give.  No header of the GPU toolchain is needed, so the host test
// compiles these very functions with g++.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define ABL_RR_FN __host__ __device__ __forceinline__
#else
#define ABL_RR_FN inline
#endif

namespace abl {

// sqrt(f) correctly rounded, given a root s within one unit in the last place u,
// for f from 2^-96 up.  Tuckerman's test (R. C. Agarwal et al., IBM J. Res. Dev.
// 30(2), 1986, pp. 126-144): d = s - u is nearer exactly when f <= s * d, since the
// midpoint's square is s * d + u^2 / 4, and f and s * d are multiples of u^2 (an ulp
// of f is at least 2^23 u^2); likewise s + u is nearer exactly when f > s * (s + u).
// Each product is compared through the sign of one fma.  Zero, infinity and NaN
// come through as they are.
ABL_RR_FN float root_from(float f, float s) {
  const uint32_t sb = __builtin_bit_cast(uint32_t, s);
  const float below = __builtin_bit_cast(float, sb - 1u), above = __builtin_bit_cast(float, sb + 1u);
  float r = s;
  if (__builtin_fmaf(-below, s, f) <= 0.f) r = below;
  if (__builtin_fmaf(-above, s, f) > 0.f) r = above;
  return r;
}

// 1 / b in double, given a float reciprocal y0 within a relative 2^-22, for 2^-100 <=
// |b| <= 2^100, correctly rounded and also so when rounded to float.  Two
// Newton-Raphson steps (relative error 2^-44, then the rounding): 1 - b y is exact
// in the fma for a 24-bit b, so the last step rounds (1/b)(1 - 2^-88), and 1/b is no
// nearer than 2^-77 to a midpoint of doubles (b m - 1 is a non-zero multiple of 2^-76
// for a midpoint m) and no nearer than 2^-48 to one of floats.
ABL_RR_FN double rcp_from(float b, float y0) {
  const double B = (double) b;
  double y = (double) y0;
  y = __builtin_fma(y, __builtin_fma(-B, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-B, y, 1.0), y);
  return y;
}

}  // namespace abl
