/* Host-side check of the zero-point code rule without a division (hyc_code_zp_word) against the rule with one
 * (hyc_code_from_t_exact of x / s + z): for every significand of the step over a spread of its exponents, every one of the 65536 bf16
 * inputs (NaNs and infinities included) and a set of zero points - the small integers that the calibration leaves, fractions
 * whose sums fall next to ties, large and tiny ones up to the limit - the codes must be equal at 2, 4 and 8 bits.
 * Prints the number of triples and of mismatches; exit status 0 iff none.
 *
 * Build (done by the test that runs it):
 *   gcc -O2 -fopenmp -ffp-contract=off -I<package>/csrc check_zp_code.c -lm
 */
#include <stdio.h>
#include "hyc_quant_math.h"

static float bf16(float f) { return hyc_bf16_to_f32(hyc_f32_to_bf16(f)); }

int main(void) {
    static const float zs[] = {0.0f, -0.0f, 1.0f, -1.0f, 3.0f, -7.0f, 127.0f, -128.0f, 0.5f, -0.5f, 0.25f, 1.5f, -2.5f, 0.49804688f, -0.33203125f, 100.5f,
                               1e-3f, -1e-20f, 1e-38f, 1e5f, -3e9f, 1.8e19f, -1.8e19f};
    static const int exps[] = {68, 100, 118, 120, 122, 124, 126, 127, 128, 130, 160, 186};
    unsigned long long triples = 0, bad = 0;
#pragma omp parallel for collapse(2) schedule(dynamic, 8) reduction(+ : triples, bad)
    for (int e = 0; e < (int)(sizeof exps / sizeof exps[0]); ++e)
        for (int m = 0; m < 128; ++m) {
            const float s = hyc_bf16_to_f32((uint16_t)(exps[e] << 7 | m));
            if (!hyc_scale_is_fast(s)) continue;
            const float y = HYC_ZP_SCALE / s, s16 = s / HYC_ZP_SCALE;
            for (unsigned xb = 0; xb < 65536u; xb += 1) {
                const float x = hyc_bf16_to_f32((uint16_t)xb), quotient = x / s;
                for (int k = 0; k < (int)(sizeof zs / sizeof zs[0]); ++k) {
                    const float z = bf16(zs[k]);
                    if (!(fabsf(z) <= HYC_ZP_MAX)) continue;
                    ++triples;
                    for (int q = 2; q <= 8; q *= 2) {
                        const int want = hyc_code_from_t_exact(quotient + z, q);
                        if (((hyc_code_zp_word(x, y, s16, z * HYC_ZP_SCALE, q) >> 16) & 0xff) != want) {
                            ++bad;
                            if (bad < 3) printf("x=%a s=%a z=%a bits=%d\n", x, s, z, q);
                        }
                    }
                }
            }
        }
    printf("triples=%llu mismatches=%llu\n", triples, bad);
    return bad ? 1 : 0;
}
