// root_from and rcp_from (openabl_amd/csrc/abl_root_rcp.hpp, compiled here as they
// are) with the instruction's root and reciprocal replaced by every value within
// one unit in the last place of the true one, against the IEEE root and divisions.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "abl_root_rcp.hpp"

static uint32_t bits_of(float f) { return __builtin_bit_cast(uint32_t, f); }
static float of_bits(uint32_t u) { return __builtin_bit_cast(float, u); }
static uint64_t state = 88172645463325252ull;
static uint64_t draw() {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state;
}

int main(int argc, char **argv) {
  const long n = argc > 1 ? atol(argv[1]) : 1000000;
  long bad = 0;
  for (long k = 0; k < n; k++) {
    // exponents -96..127, mantissas at random, near the ends, and squares of
    // midpoints, where the root is hardest to round
    uint32_t u = ((uint32_t) (31 + draw() % 223) << 23) | (uint32_t) (draw() & 0x7FFFFF);
    if (k % 4 == 1) u = (u & 0x7F800000u) | (uint32_t) (draw() % 16);
    if (k % 4 == 2) u = (u & 0x7F800000u) | (0x7FFFFFu - (uint32_t) (draw() % 16));
    if (k % 4 == 3) {
      const double m = 1.0 + ((double) (draw() & 0x7FFFFF) + 0.5) * 0x1p-23;
      u = bits_of((float) (m * m));
    }
    const float f = of_bits(u);
    const float want = std::sqrt(f);
    for (int d = -1; d <= 1; d++)
      bad += abl::root_from(f, of_bits(bits_of(want) + (uint32_t) d)) != want;
    if (f >= 0x1p-95f && f <= 0x1p95f) {
      const float y = 1.0f / f;
      for (int d = -1; d <= 1; d++) {
        const double r = abl::rcp_from(f, of_bits(bits_of(y) + (uint32_t) d));
        bad += r != 1.0 / (double) f;
        bad += (float) r != y;
      }
    }
  }
  // what the root's instruction returns for them comes through
  for (const float f : {0.0f, -0.0f, INFINITY}) bad += bits_of(abl::root_from(f, f)) != bits_of(f);
  bad += !std::isnan(abl::root_from(NAN, NAN));
  std::printf("%ld wrong of %ld\n", bad, n);
  return bad ? 1 : 0;
}
