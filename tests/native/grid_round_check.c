/*
 * Exhaustive proof, on the CPU, of the two-operation rounding the fused quantisers use for rows (columns) whose scale is a normal
 * fp16 number.  There s = fp16(absmax / 127) and |x| <= absmax, so the quotient stays within 127.07; it is a tie exactly or at
 * least 2^-12 away from one, and a first rounding of x * (1 / s) to the grid of 2^-12 keeps every case what it is:
 *
 *     reference:  n = int8(rint(x / s))                          (IEEE fp32 divide, cuda/gemm.cu:16)
 *     fast:       y = 1/s;  q = fma(x, y, 3072);  n = low byte of the bit pattern of (q + 12579840)
 *
 * for EVERY finite fp16 absmax with a normal scale and EVERY fp16 x with |x| <= absmax, and every fp16 NaN x (0 either way).
 * The pairs depend on absmax through s alone: each scale is checked once, over the x of its largest absmax.  Prints the number of
 * mismatching pairs; exits non-zero if any.
 */
#include <immintrin.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

int main(void) {
    static uint16_t largest[0x7c00];       /* by scale: its largest absmax, 0 if it is the scale of none */
    for (int a = 1; a < 0x7c00; ++a) {
        const uint16_t sb = _cvtss_sh(_cvtsh_ss((uint16_t)a) / 127.0f, 0);       /* to nearest even */
        if (sb >= 0x0400 && sb <= 0x7bff) largest[sb] = (uint16_t)a;
    }
    long long bad = 0, pairs = 0, scales = 0;
#pragma omp parallel for schedule(dynamic, 64) reduction(+ : bad, pairs, scales)
    for (int si = 0x0400; si < 0x7c00; ++si) {
        if (!largest[si]) continue;
        const float s = _cvtsh_ss((uint16_t)si);
        const float y = 1.0f / s;
        ++scales;
        for (int xi = 0; xi < 65536; ++xi) {
            const int mag = xi & 0x7fff;
            if (mag > largest[si] && mag <= 0x7c00) continue;
            const float x = _cvtsh_ss((uint16_t)xi), d = x / s;
            const int ref = d != d ? 0 : (int)rintf(d);
            volatile float q = fmaf(x, y, 3072.0f);
            volatile float t = q + 12579840.0f;
            const float tt = t;
            uint32_t b;
            memcpy(&b, &tt, 4);
            const int fast = (int)(int8_t)(b & 0xffu);
            if (ref < -128 || ref > 127 || ref != fast) {
                if (bad < 5) fprintf(stderr, "mismatch x=%04x s=%04x ref=%d fast=%d\n", xi, si, ref, fast);
                ++bad;
            }
            ++pairs;
        }
    }
    printf("%lld scales, %lld pairs, %lld mismatches\n", scales, pairs, bad);
    return bad != 0;
}
