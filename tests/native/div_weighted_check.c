/* x / c by the corrected product the multigrid tail uses (q0 = x r, e = x - q0
 * c, q = q0 + e r, r = RN(1/c)) against IEEE division, for every count c =
 * fluid + w outside with w = 2 2^l / (2^l + 1), l = 1 .. 11, and x = m 2^k
 * with every 24-bit mantissa on a stride, exponents 2^-100, 2^-99, 1 and
 * 2^127: the range in which the fast form stands alone is |x| >= 2^-100, and
 * scaling x by a power of two changes nothing between.  `stride` 1 covers all
 * mantissas.  Prints the number of counts and of mismatches. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

int main(int argc, char **argv) {
  const uint32_t stride = argc > 1 ? (uint32_t)atoi(argv[1]) : 61;
  const int ex[4] = {-100, -99, 0, 127};
  long bad = 0, counts = 0;
  for (int l = 1; l <= 11; l++) {
    const float w = (float)(2.0 * ldexp(1.0, l) / (ldexp(1.0, l) + 1.0));
    for (int fl = 0; fl <= 6; fl++)
      for (int out = 0; out <= 5 && fl + out <= 6; out++) {
        if (fl + out == 0) continue;
        volatile float wo = w * (float)out;
        const float c = (float)fl + wo, r = 1.0f / c;
        counts++;
        for (int k = 0; k < 4; k++)
          for (uint32_t m = 0; m < (1u << 23); m += stride) {
            const float x = ldexpf(1.0f + (float)m * 0x1p-23f, ex[k]);
            const float q0 = x * r;
            const float e = fmaf(-q0, c, x);
            bad += fmaf(e, r, q0) != x / c;
          }
      }
  }
  printf("%ld %ld\n", counts, bad);
  return bad != 0;
}
