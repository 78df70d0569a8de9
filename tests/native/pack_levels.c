/* Exhaustive check of the INT4 pack's level arithmetic (csrc/int4_pack.hip, pack_levels) against the
 * IEEE quotient: rint(q) = rint(RN(x / s)) with y = RN(1 / s), q0 = RN(x y),
 * q = RN(q0 + RN(x - q0 s) y).
 *
 * |q - x / s| is below 0.51 ulp (q0 is within 1.5 ulp of x / s and y within 2^-24 relative of
 * 1 / s), so the two integers can only differ where x / s lies within 2 ulps of a half-integer
 * h = 0.5, 1.5, ..., 7.5 (|x| <= absmax and s >= RN(absmax / 7) bound |x / s| by 7.0000005). Powers of two do not
 * matter away from overflow and underflow (s >= 1e-8; quotients below 1/4 round to 0 either way),
 * so it is enough to take x in [1, 2) and, for each h, the scales next to x / h: one ulp of s moves
 * the quotient by at least half an ulp, so eight on each side cover the 2 ulps. Prints the number of
 * pairs and of mismatches. The argument is a stride over the mantissas (1 = all of them).
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static float f_of(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t u_of(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

int main(int argc, char** argv) {
  const int stride = argc > 1 ? atoi(argv[1]) : 1;
  long long pairs = 0, bad = 0;
#pragma omp parallel for reduction(+ : pairs, bad) schedule(static)
  for (long long m = 0; m < (1 << 23); m += stride) {
    const float x = f_of(0x3f800000u + (uint32_t)m);
    for (int j = 0; j < 8; ++j) {
      const float mid = (float)((double)x / (j + 0.5));
      for (int d = -8; d <= 8; ++d) {
        const float s = f_of(u_of(mid) + (uint32_t)d);
        const float y = 1.0f / s;
        const float q0 = x * y;
        const float q = fmaf(fmaf(-q0, s, x), y, q0);
        const float k = (q + 12582912.0f) - 12582912.0f;
        ++pairs;
        if (k != rintf(x / s)) ++bad;
      }
    }
  }
  printf("pairs=%lld bad=%lld\n", pairs, bad);
  return bad != 0;
}
