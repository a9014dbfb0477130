/*
 * The division of the backward quantisers, on the CPU.  They round products of two fp16 numbers by a scale of the data's own that is
 * an fp32 number,
 *     s = fp32(absmax / 127),   |x| <= absmax,
 * and divide through the reciprocal with two residual steps:
 *
 *     reference:  n = int8(rint(x / s))                          (IEEE fp32 divide, cuda/gemm.cu:139-172)
 *     fast:       y = 1/s;  q0 = x*y;  q1 = fma(fma(-s, q0, x), y, q0);  q2 = fma(fma(-s, q1, x), y, q1);
 *                 n = low byte of the bit pattern of (q2 + 12582912.0f)
 *
 * q2 is to be the correctly rounded quotient, and n its nearest integer.  Checked for EVERY significand an absmax can have (products of
 * two 11-bit integers; powers of two scale every step alike) and, for each of its scales, the fp32 numbers around every boundary
 * between two integers, (k + 1/2) * s and three to either side, among them every product that lies so close; the absmax itself; and NaN.
 * Prints the number of mismatches; exits non-zero if any.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static int check(float x, float s, float y, float top) {
    if (!(x <= top) && x == x) return 0;
    const float d = x / s;
    const int ref = d != d ? 0 : (int)rintf(d);
    const float q0 = x * y;
    const float q1 = fmaf(fmaf(-s, q0, x), y, q0);
    const float q2 = fmaf(fmaf(-s, q1, x), y, q1);
    volatile float t = q2 + 12582912.0f;
    const float tt = t;
    uint32_t b;
    memcpy(&b, &tt, 4);
    return (int)(int8_t)(b & 0xffu) != ref || (d == d && q2 != d);
}

int main(void) {
    static uint8_t seen[1 << 22];            /* products of two significands, 2^20 ... (2^11 - 1)^2, by value */
    for (uint32_t a = 1024; a < 2048; ++a)
        for (uint32_t b = a; b < 2048; ++b) seen[a * b] = 1;
    long long bad = 0, pairs = 0, scales = 0;
#pragma omp parallel for schedule(dynamic, 4096) reduction(+ : bad, pairs, scales)
    for (uint32_t p = 1 << 20; p < 1 << 22; ++p) {
        if (!seen[p]) continue;
        const float top = (float)p;
        const float s = (float)((double)top / 127.0);
        const float y = 1.0f / s;
        ++scales;
        for (int k = 0; k < 127; ++k) {
            float x = (float)(((double)k + 0.5) * (double)s);
            for (int i = 0; i < 3; ++i) x = nextafterf(x, 0.0f);
            for (int i = 0; i < 7; ++i, x = nextafterf(x, INFINITY)) {
                bad += check(x, s, y, top);
                ++pairs;
            }
        }
        bad += check(top, s, y, top) + check(NAN, s, y, top);
        pairs += 2;
    }
    printf("%lld scales, %lld pairs, %lld mismatches\n", scales, pairs, bad);
    return bad != 0;
}
