/* fd2_div_by (fd2_math.h) on every quotient it could round wrongly (test
 * infrastructure; prints the number of wrong results, 0 expected).
 *
 * With y the correctly rounded 1/b and q = a y rounded, r = a - b q is exact
 * and q + r y differs from a/b by less than 2^-23 ulp before its rounding, so
 * the result can only be wrong where a/b lies that close to the midpoint of
 * two floats.  For 24-bit significands a, b in [2^23, 2^24) the midpoints are
 * M/2^24 (a >= b) or M/2^25 (a < b) with M odd in [2^24, 2^25), and
 * a 2^s = M b + k at a distance of |k|/(2b) ulp, so |k| <= 3 covers them.  For
 * every b and k the congruence M b = -k (mod 2^s) gives the candidates. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>

/* 1/b mod 2^64 of an odd b (Newton's iteration doubles the correct bits) */
static uint64_t inverse(uint64_t b) {
  uint64_t x = b;
  for (int i = 0; i < 6; ++i) x *= 2 - b * x;
  return x;
}

int main(void) {
  unsigned long long n = 0, wrong = 0;
  for (uint64_t b = 1u << 23; b < 1u << 24; ++b) {
    const int t = __builtin_ctzll(b);
    const uint64_t inv = inverse(b >> t);
    const float fb = (float)b, y = 1.0f / fb;
    for (int s = 24; s <= 25; ++s)
      for (int k = -3; k <= 3; ++k) {
        if (k == 0 || t > s || k % (1 << t) != 0) continue;
        const uint64_t step = (uint64_t)1 << (s - t);
        uint64_t m = ((uint64_t)(int64_t)(-(k / (1 << t))) * inv) & (step - 1);
        for (; m < (uint64_t)1 << 25; m += step) {
          if (m < (uint64_t)1 << 24 || !(m & 1)) continue;
          const uint64_t a = (uint64_t)((int64_t)(m * b) + k) >> s;
          if (a < 1u << 23 || a >= 1u << 24 || (s == 24 ? a < b : a >= b)) continue;
          ++n;
          const float fa = (float)a, q = fa * y;
          if (fmaf(fmaf(-fb, q, fa), y, q) != fa / fb) ++wrong;
        }
      }
  }
  printf("%llu quotients near a midpoint, %llu wrong\n", n, wrong);
  return wrong != 0 || n < 1000000;
}
