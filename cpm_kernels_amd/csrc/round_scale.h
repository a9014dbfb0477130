// The int8 values of a gradient times the other operand's scales, with a scale per row (cu_gemm_backward_round_scale, cuda/gemm.cu:100-137), for rows that a
// wave holds in registers.
#pragma once
#include "common.h"
#include <type_traits>

namespace cpmk {

struct RoundScaleArgs {
    const half_t *mat, *scale_y;   // (batch, n, m); (batch, m), or (m) shared by the batch (bc)
    int8_t* out;                   // (batch, n, ld): past the matrix's columns zeros
    half_t* scale_x;               // (batch, n)
    int64_t rows;                  // batch * n
    int32_t n, m;
    int bc;
    int32_t ld;
    uint32_t first;                // number of the first workgroup of the rows, in a launch that they share
};

// eight products x * sy rounded to multiples of s (own: s is the data's own and in the range of the short sequence)
__device__ __forceinline__ uint2_t round8_own_scale(half8_t x, half8_t sy, float s, float y, bool own) {
    int32_t t[8];
    if (own) {
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = (int32_t)quant_i8_own_fp32_scale_bits((float)x[e] * (float)sy[e], s, y);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = quant_i8((float)x[e] * (float)sy[e], s);
    }
    return uint2_t{pack4_i8(t[0], t[1], t[2], t[3]), pack4_i8(t[4], t[5], t[6], t[7])};
}

// Rows of at most 2048 columns, kept in registers: a wave takes U consecutive rows of P 16-byte pieces
// per lane (P * U = 4 loads in flight per lane, the matrix read once, NTH with the non-temporal hint), finds each
// row's maximum over the wave with data-parallel-primitive operands and rounds from the registers.
// UA: rows that are not whole 16-byte pieces or buffers off 16-byte boundaries -- a piece inside its row still comes in
// one 16-byte load and leaves in one 8-byte store (global accesses need no alignment), the piece across a row's end
// is read with what lies behind it and leaves in at most three narrower accesses.
// The two rounding sequences are chosen once for the wave's rows: a choice per row kept their chains from running side by side (780 rows
// of 24 6.9 us, 4.7 so; 20000 of 512 11.1 -> 8.1; 81920 of 512 30 -> 23.5, 5.3 TB/s).
template <int P, int U, bool UA, bool NTH>
__device__ __forceinline__ void round_scale_rows_reg(const RoundScaleArgs& a, int64_t wave) {
    const int64_t rows = a.rows;
    const int32_t n = a.n, m = a.m, ld = a.ld;
    const int lane = threadIdx.x & 63;
    const int64_t row0 = wave * U;
    if (row0 >= rows) return;
    half8_t xv[U][P], sv[U][P];
    const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    // UA: every load is made (pieces past a row's end as its first one) and put right behind them all: a row's end lies in every wave, and under conditions of their own the loads
    // waited for one another (4 x 10240 rows of 500 33 -> 26 us, 4 x 896 of 172 9.6 -> 8.0).  Rows of less than a piece take the conditions.
    const int64_t last_x = rows * m - 8, last_s = (a.bc ? 1 : rows / n) * (int64_t)m - 8;
    const bool pieces = !UA || m >= 8;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t row = row0 + u < rows ? row0 + u : rows - 1;
        const int64_t x0 = row * m, s0 = a.bc ? 0 : (row / n) * m;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int32_t j = lane * 8 + p * 512;
            if constexpr (UA) {
                if (pieces) {
                    xv[u][p] = half8_unset();
                    sv[u][p] = half8_unset();
                    if (j < m) {
                        xv[u][p] = load_half8_any(a.mat + min(x0 + j, last_x));
                        sv[u][p] = load_half8_any(a.scale_y + min(s0 + j, last_s));
                    }
                } else {
                    xv[u][p] = j < m ? load_half8_head_any(a.mat + x0, m, zero) : zero;
                    sv[u][p] = j < m ? load_half8_head_any(a.scale_y + s0, m, zero) : zero;
                }
            } else {
                xv[u][p] = sv[u][p] = zero;
                if (j < m) {
                    const half8_t* src = reinterpret_cast<const half8_t*>(a.mat + x0 + j);
                    xv[u][p] = NTH ? __builtin_nontemporal_load(src) : *src;
                    sv[u][p] = *reinterpret_cast<const half8_t*>(a.scale_y + s0 + j);
                }
            }
        }
    }
    if (UA && pieces) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t row = row0 + u < rows ? row0 + u : rows - 1;
            // (its last piece ends behind the buffer's in the last row alone, rows are a piece and more; looked for at each piece the short rows paid: 240600 of 12 82 us, 60 so)
            const bool end_x = row + 1 == rows, end_s = a.bc || row >= rows - n;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int32_t j = lane * 8 + p * 512;
                if (j + 8 > m) {
                    const uint4_t keep = half8_keep(m - j);
                    if (end_x && j < m) xv[u][p] = half8_down(xv[u][p], j + 8 - m);
                    if (end_s && j < m) sv[u][p] = half8_down(sv[u][p], j + 8 - m);
                    xv[u][p] = half8_fill(xv[u][p], keep, zero);
                    sv[u][p] = half8_fill(sv[u][p], keep, zero);
                }
            }
        }
    }
    float s[U];
    bool own = true;        // (the same for the whole wave)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        float mx = 0.0f;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(fabsf((float)xv[u][p][e] * (float)sv[u][p][e]), mx);
        mx = __builtin_bit_cast(float, wave_max_u32_uniform(__builtin_bit_cast(uint32_t, mx)));      // (non-negative floats order as their bits)
        s[u] = (float)((double)mx / 127.0);
        own = own && own_scale_in_range(s[u]);
        if (lane == 0 && row0 + u < rows) a.scale_x[row0 + u] = (half_t)s[u];
    }
    auto finish = [&](auto ownc) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t row = row0 + u;
            if (row >= rows) break;
            const float y = 1.0f / s[u];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int32_t j = lane * 8 + p * 512;
                if (j < ld) {        // (past the end of the row: zeros)
                    const uint2_t w = round8_own_scale(xv[u][p], sv[u][p], s[u], y, decltype(ownc)::value);
                    int8_t* dst = a.out + row * ld + j;
                    if constexpr (!UA) {
                        *reinterpret_cast<uint2_t*>(dst) = w;
                    } else if (j + 8 <= ld) {
                        store_byte8_any(dst, w.x, w.y);
                    } else {
                        store_byte8_head_any(dst, ld & 7, w.x, w.y);
                    }
                }
            }
        }
    };
    if (own) finish(std::true_type{});
    else finish(std::false_type{});
}

}  // namespace cpmk
