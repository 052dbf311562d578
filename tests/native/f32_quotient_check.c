/* The kernels' float32 quotient x / s from r = RN(1 / s) (csrc/scale_quotient.h,
 * scale_quotient) against the IEEE division, bit for bit where |x / s| >= 2^-12 and
 * below that within 2^-11: random scales over the declared range, and for each the
 * numerators around every half-integer quotient (where a code changes), random ones
 * and tiny ones. "uncorrected" as argument keeps the bare product. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static uint64_t next(uint64_t* st) {
  uint64_t z = (*st += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static float fbits(uint32_t b) { float f; memcpy(&f, &b, 4); return f; }

static float quotient(float x, float s, float r, int bare) {
  const float q0 = x * r;
  const float q1 = fmaf(fmaf(-q0, s, x), r, q0);
  return bare ? q0 : fmaf(fmaf(-q1, s, x), r, q1);
}

int main(int argc, char** argv) {
  const int bare = argc > 1 && !strcmp(argv[1], "uncorrected");
  unsigned long long n = 0, bad = 0;
#pragma omp parallel for reduction(+ : n, bad)
  for (int i = 0; i < 300000; ++i) {
    uint64_t st = 77 + (uint64_t)i * 1000003;
    const uint64_t z = next(&st);
    const int ex = 127 - 30 + (int)((z >> 32) % (30 + 121));          /* 2^-30 <= s < 2^121 */
    const float s = fbits(((uint32_t)ex << 23) | (uint32_t)(z & 0x7FFFFF)), r = 1.0f / s;
    for (int k = 0; k < 600; ++k) {
      const uint64_t y = next(&st);
      float x;
      if (k < 512) {                                                  /* half-integers and their neighbours */
        x = (float)(k / 4) * s + 0.5f * s;
        const int ulps = (int)(y % 7) - 3;
        uint32_t b; memcpy(&b, &x, 4); x = fbits(b + (uint32_t)ulps);
      } else if (k < 590) {
        x = (float)((double)(y >> 11) * 0x1p-53 * 127.0 * s);
      } else {
        x = fbits((uint32_t)(y % 0x30000000u));                       /* subnormal to 2^-31 */
        if (x > 127.0f * s) continue;
      }
      if (y >> 63) x = -x;
      const float want = x / s, got = quotient(x, s, r, bare);
      ++n;
      if (fabsf(want) >= 0x1p-12f) bad += memcmp(&want, &got, 4) != 0;
      else bad += !(fabsf(got) < 0x1p-11f);
    }
  }
  printf("checked %llu mismatches %llu\n", n, bad);
  return bad != 0;
}
