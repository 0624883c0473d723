/* The quotient of the iteration kernels (p2_recip, p2_recip_wide, p2_quotient in poker2_amd/csrc/common.h) in the C
 * library's fused multiply-add, against the C division: every mantissa of the divisor, some dividends for each of them,
 * among them those whose quotient lies next to the middle between two floats, and every reciprocal that hardware within
 * one unit in the last place may start from. */
#include <math.h>
#include <stdint.h>
#include <string.h>

static float from_bits(uint32_t u) {
  float x;
  memcpy(&x, &u, 4);
  return x;
}
static uint32_t bits_of(float x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  return u;
}
static uint64_t draw(uint64_t* s) {                        /* splitmix64 */
  uint64_t z = (*s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

static float rcp(float b, int ulps) { return from_bits(bits_of((float)(1.0 / (double)b)) + (uint32_t)ulps); }
static float recip(float b, int ulps) {
  const float y = rcp(b, ulps);
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
static float recip_wide(float b, int ulps) {
  const float y = rcp(b * 0x1p-32f, ulps) * 0x1p-32f;
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
static float quotient(float a, float b, float y) {
  const float q = a * y;
  return fmaf(fmaf(-b, q, a), y, q);
}

/* Quotients that differ from a / b, for divisors of exponent `eb` (every `step`-th mantissa) and dividends of exponent
 * `ea`; `worst`: the largest difference in units of the last place.  Finite operands: the special ones are what
 * v_div_fixup_f32 defines. */
int64_t p2o_quotient_differs(int eb, int ea, int wide, int64_t step, int dividends, int64_t* worst) {
  int64_t differ = 0, most = 0;
#pragma omp parallel for reduction(+ : differ) reduction(max : most)
  for (int64_t m = 0; m < (1 << 23); m += step) {
    const float b = ldexpf(from_bits(0x3F800000u | (uint32_t)m), eb);
    uint64_t s = (uint64_t)m * 977 + 13;
    float y[3];
    for (int d = 0; d < 3; ++d) y[d] = wide ? recip_wide(b, d - 1) : recip(b, d - 1);
    for (int k = 0; k < dividends; ++k) {
      uint32_t am = (uint32_t)(draw(&s) & 0x7FFFFF);
      if (k & 1) {                                         /* the float nearest to b times a middle between two floats */
        const double middle = 1.0 + ((double)am + 0.5) * 0x1p-23;
        am = bits_of((float)((double)from_bits(0x3F800000u | (uint32_t)m) * middle)) & 0x7FFFFF;
      }
      const float a = ldexpf(from_bits(0x3F800000u | am), ea), want = a / b;
      for (int d = 0; d < 3; ++d) {
        const float got = quotient(a, b, y[d]);
        if (bits_of(got) == bits_of(want)) continue;
        int64_t off = (int64_t)bits_of(got) - (int64_t)bits_of(want);
        if (off < 0) off = -off;
        if (off > most) most = off;
        ++differ;
      }
    }
  }
  *worst = most;
  return differ;
}
