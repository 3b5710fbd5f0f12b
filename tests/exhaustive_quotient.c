// Exhaustive check of the quotient and the rounding the activation quantizers use (csrc/quant.hip): for every fp16
// absmax a >= 0 and every fp16 x with |x| <= a, with r = 1 / scale and l = fma(-scale, r, 1) * r (r + l is 1 / scale to
// twice the precision), fma(x, r, x * l) equals the correctly rounded x / scale (the oracle's division), for
// scale = max(a / 127, 1e-30) (int8 codes) and scale = max(a, 1e-10) / 7 (int4 codes); and for the int8 quotients
// floor(q + 0.5) is the same with the sum rounded to fp32 (the oracle's) and in exact arithmetic, so that one
// conversion may do both steps in either way. The quotient is odd in x; the rounding is checked for both signs.
// Build: gcc -O2 -fopenmp -ffp-contract=off exhaustive_quotient.c -lm. Exit status 0 when nothing differs.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
static float h2f(uint16_t h) {  // h >= 0, finite
    const int e = h >> 10, m = h & 1023;
    return e == 0 ? ldexpf((float)m, -24) : ldexpf((float)(m | 1024), e - 25);
}
int main(void) {
    static float value[0x7c00];
    for (int i = 0; i < 0x7c00; i++) value[i] = h2f((uint16_t)i);
    long quotient8 = 0, quotient4 = 0, rounding = 0;
    #pragma omp parallel for reduction(+:quotient8, quotient4, rounding) schedule(dynamic, 64)
    for (int ha = 0; ha < 0x7c00; ha++) {
        const float a = value[ha];
        const float s8 = fmaxf(a / 127.f, 1e-30f), r8 = 1.f / s8, l8 = fmaf(-s8, r8, 1.f) * r8;
        const float s4 = fmaxf(a, 1e-10f) / 7.f, r4 = 1.f / s4, l4 = fmaf(-s4, r4, 1.f) * r4;
        for (int hx = 0; hx <= ha; hx++) {
            const float x = value[hx], q = x / s8;
            quotient8 += q != fmaf(x, r8, x * l8);
            quotient4 += x / s4 != fmaf(x, r4, x * l4);
            rounding += floorf(q + 0.5f) != (float)floor((double)q + 0.5);
            rounding += floorf(-q + 0.5f) != (float)floor(-(double)q + 0.5);
        }
    }
    printf("mismatches: int8 quotient %ld, int4 quotient %ld, rounding %ld\n", quotient8, quotient4, rounding);
    return quotient8 || quotient4 || rounding;
}
