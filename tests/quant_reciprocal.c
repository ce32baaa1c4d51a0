/* Exhaustive check of the prompt quantizers' code arithmetic (iq_quantize.h).
 * For every pair of finite operands x >= 0, s > 0 of the activation type, every
 * level count L in {15, 7, 3, 1} and every r within one fp32 ulp of 1/s,
 *     rint(min(RN(RN32(x r)), L)) == rint(min(RN(RN32(x / s)), L))
 * where RN rounds to fp16, or to bf16 with s in [2^-100, 2^100]; and the
 * scales: RN(v / L) == RN(v RN32(1/L)) for every v >= 0 of the type.
 * argv[1] = step: every step-th s (1: all).  Prints the mismatch counts; exits
 * 1 on any. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static float fb(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

/* x >= 0 rounded to fp16 (nearest, ties to even), as fp32 */
static float rn16(float x) {
  if (x >= 65520.0f) return INFINITY;
  if (x < 0x1p-14f) return (x + 0x1.8p-1f) - 0x1.8p-1f; /* subnormal: ulp 2^-24 */
  const uint32_t u = bits(x);
  return fb((u + 0xfffu + ((u >> 13) & 1u)) & ~0x1fffu);
}
static float rnbf(float x) {
  const uint32_t u = bits(x);
  if (u >= 0x7f800000u) return x;
  return fb((u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u);
}
static float f16v(uint32_t h) {
  const uint32_t e = h >> 10, m = h & 0x3ff;
  return e ? ldexpf((float)(m | 0x400), (int)e - 25) : ldexpf((float)m, -24);
}
static float code(float y, float L) { return rintf(y < L ? y : L); }

int main(int argc, char** argv) {
  const int step = argc > 1 ? atoi(argv[1]) : 1;
  static const float Ls[4] = {15.f, 7.f, 3.f, 1.f};
  static float v16[0x7c00], vbf[0x7f80];
  long long bad16 = 0, badbf = 0, bads = 0;
  for (uint32_t h = 0; h < 0x7c00; ++h) v16[h] = f16v(h);
  for (uint32_t h = 0; h < 0x7f80; ++h) vbf[h] = fb(h << 16);
  for (int k = 0; k < 4; ++k) {
    const float L = Ls[k], rl = 1.0f / L;
    for (int h = 0; h < 0x7c00; ++h) bads += rn16(v16[h] / L) != rn16(v16[h] * rl);
    for (int h = 0; h < 0x7f80; ++h) bads += rnbf(vbf[h] / L) != rnbf(vbf[h] * rl);
  }
#pragma omp parallel for schedule(dynamic, 16) reduction(+ : bad16, badbf)
  for (int j = 1; j < 0x7f80; j += step) {
    if (j < 0x7c00) {
      const float s = v16[j], r = 1.0f / s, rr[3] = {fb(bits(r) - 1), r, fb(bits(r) + 1)};
      for (int i = 0; i < 0x7c00; ++i) {
        const float q = rn16(v16[i] / s);
        for (int m = 0; m < 3; ++m) {
          const float p = rn16(v16[i] * rr[m]);
          if (p != q)
            for (int k = 0; k < 4; ++k) bad16 += code(p, Ls[k]) != code(q, Ls[k]);
        }
      }
    }
    const float s = vbf[j];
    if (s >= 0x1p-100f && s <= 0x1p100f) {
      const float r = 1.0f / s, rr[3] = {fb(bits(r) - 1), r, fb(bits(r) + 1)};
      for (int i = 0; i < 0x7f80; ++i) {
        const float q = rnbf(vbf[i] / s);
        for (int m = 0; m < 3; ++m) {
          const float p = rnbf(vbf[i] * rr[m]);
          if (p != q)
            for (int k = 0; k < 4; ++k) badbf += code(p, Ls[k]) != code(q, Ls[k]);
        }
      }
    }
  }
  printf("fp16 %lld bf16 %lld scales %lld\n", bad16, badbf, bads);
  return bad16 || badbf || bads;
}
