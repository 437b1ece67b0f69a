/* sqrt_rn_f32 and rcp_rn (openabl_amd/csrc/abl_device.hpp) restated in C with
 * the hardware's root and reciprocal replaced by every value within one unit
 * in the last place of the true one, against the IEEE root and divisions. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint32_t bits_of(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}
static float of_bits(uint32_t u) {
  float f;
  memcpy(&f, &u, 4);
  return f;
}
static uint64_t state = 88172645463325252ull;
static uint64_t draw(void) {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state;
}

/* s: a root of f within one ulp */
static float root(float f, float s) {
  const float below = of_bits(bits_of(s) - 1u), above = of_bits(bits_of(s) + 1u);
  float r = s;
  if (fmaf(-below, s, f) <= 0.f) r = below;
  if (fmaf(-above, s, f) > 0.f) r = above;
  return r;
}

/* y0: a float reciprocal of b within one ulp */
static double recip(float b, float y0) {
  const double B = (double) b;
  double y = (double) y0;
  y = fma(y, fma(-B, y, 1.0), y);
  y = fma(y, fma(-B, y, 1.0), y);
  return y;
}

int main(int argc, char **argv) {
  const long n = argc > 1 ? atol(argv[1]) : 1000000;
  long bad = 0;
  for (long k = 0; k < n; k++) {
    /* exponents -96..127, mantissas at random, near the ends, and squares of
     * midpoints, where the root is hardest to round */
    uint32_t u = ((uint32_t) (31 + draw() % 223) << 23) | (uint32_t) (draw() & 0x7FFFFF);
    if (k % 4 == 1) u = (u & 0x7F800000u) | (uint32_t) (draw() % 16);
    if (k % 4 == 2) u = (u & 0x7F800000u) | (0x7FFFFFu - (uint32_t) (draw() % 16));
    if (k % 4 == 3) {
      const double m = 1.0 + ((double) (draw() & 0x7FFFFF) + 0.5) * 0x1p-23;
      u = bits_of((float) (m * m));
    }
    const float f = of_bits(u);
    const float want = sqrtf(f);
    for (int d = -1; d <= 1; d++) bad += root(f, of_bits(bits_of(want) + (uint32_t) d)) != want;
    if (f >= 0x1p-95f && f <= 0x1p95f) {
      const float y = 1.0f / f;
      for (int d = -1; d <= 1; d++) {
        const double r = recip(f, of_bits(bits_of(y) + (uint32_t) d));
        bad += r != 1.0 / (double) f;
        bad += (float) r != y;
      }
    }
  }
  printf("%ld wrong of %ld\n", bad, n);
  return bad ? 1 : 0;
}
