// Register-resident column tiles for reductions over dim 1 of a (batch, n, m) fp16 tensor.
//
// The reference walks such tensors with 32x32 thread blocks, 64-byte row segments and two or
// three passes over global memory (cuda/layernorm.cu:6-71, cuda/softmax.cu:6-43).  Here one
// workgroup of NT threads owns all n rows of LPR*8 adjacent columns and keeps them in
// registers, so HBM is read once and written once:
//   lane -> (cg = tid % LPR, rg = tid / LPR); pass p covers rows p*(NT/LPR) + rg;
//   each lane holds R 16-byte pieces (8 columns of R rows).
// Reductions run per lane, then over the lanes of a wave that share cg (xor butterflies on
// the lane bits above log2(LPR)), then over waves through a few hundred bytes of LDS.
#pragma once
#include "common.h"

namespace cpmk {

template <int NT, int LPR, int R>
struct ColTile {
    static constexpr int RPP = NT / LPR;       // rows per pass
    static constexpr int ROWS = RPP * R;       // rows the tile can hold
    static constexpr int COLS = LPR * 8;
    static constexpr int NW = NT / 64;
    // LDS floats needed by reduce<NV>: (NW + 1) * COLS * NV
};

// Load the tile; rows >= n and columns >= m are left as `fill` in every half.  `base` is the
// (wave-uniform) start of this batch entry; element offsets inside it are 32-bit, which lets
// the compiler address with a scalar base plus one VGPR offset instead of holding R 64-bit
// pointers across the reduction phases (callers guarantee n*m < 2^31).
//
// NTL / NTS: non-temporal loads / stores.  Only for tiles whose row segments are whole 128-byte cache
// lines (LPR == 8) and for data that is not read again soon: a segment shorter than a line is completed
// by a neighbouring workgroup, so it has to allocate in L2.
//
// UA: rows that are not whole 16-byte pieces, or buffers that are not 16-byte aligned.  A piece inside its row still
// moves as one 16-byte access (global accesses need no alignment; one that crosses a cache line costs a second
// request), the piece across a row's end in at most three narrower ones.
// LOADS: what the registers of rows past the last and of columns past the row's end hold, whose loads are not made.  kLoadsPlain (not UA): `fill`, as the
// compiler likes it, which keeps the loads of eight rows a lane together; of other tiles it let them wait for one another, with copies behind each.  kLoadsKept: `fill`, in registers that the
// compiler cannot tell apart from others.  kLoadsUnset (UA): nothing yet; fewer registers where the pieces have to be put right all the same.
// UA: tiles with rows nearly throughout make every load, those of rows past the last as the last one's, so that the first piece can be used before the last one is there.
// us, loads that waited / every load made and put right half by half / this: softmax of 1024 of 500 x 500 268 / 230 / 217, of 70 x 70 10.6 / 11.8 / 10.8, its gradient of 512 of 129 x 130 28 / 14.6 / 12.9;
// LayerNorm 672 x 30 x 847 113 / 121 / 113, its gradient 234 / 338 / 237; column scales of 1024 x 70 x 70 10.6 / 18.5 / 10.9.
constexpr int kLoadsPlain = 0, kLoadsKept = 1, kLoadsUnset = 2;
constexpr int coltile_loads(bool ua, int r, int lpr) { return ua ? kLoadsUnset : r == 8 && lpr == 8 ? kLoadsPlain : kLoadsKept; }
template <int RPP, int R>
__device__ __forceinline__ bool coltile_nearly_full(int32_t n) { return n * 8 >= RPP * R * 7; }
// coltile_request makes the loads and coltile_settle puts what they brought right: a kernel of two tiles requests both before it settles one.
template <int NT, int LPR, int R, bool NTL = false, bool UA = false, int LOADS = coltile_loads(UA, R, LPR)>
__device__ inline void coltile_request(half8_t (&v)[R], const half_t* base, int32_t n, int32_t m, int32_t col0,
                                       half_t fill) {
    constexpr int RPP = NT / LPR;
    const int rg = threadIdx.x / LPR;
    const uint32_t off0 = (uint32_t)rg * (uint32_t)m + (uint32_t)col0, stride = (uint32_t)RPP * (uint32_t)m;
    half8_t none;
#pragma unroll
    for (int e = 0; e < 8; ++e) none[e] = fill;
    if constexpr (LOADS == kLoadsPlain) {
        static_assert(!UA, "whole pieces");
#pragma unroll
        for (int p = 0; p < R; ++p) {
            half8_t x = none;
            if (p * RPP + rg < n && col0 < m) {
                const half8_t* src = reinterpret_cast<const half8_t*>(base + (off0 + p * stride));
                x = NTL ? __builtin_nontemporal_load(src) : *src;
            }
            v[p] = x;
        }
        return;
    }
    const uint32_t last = (uint32_t)n * (uint32_t)m - 8u;
    if (UA && (uint32_t)n * (uint32_t)m < 8u) {        // a matrix of less than a piece: as the end of one
        half8_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = base[max(e + n * m - 8, 0)];
#pragma unroll
        for (int p = 0; p < R; ++p) v[p] = x;
        return;
    }
    auto load = [&](uint32_t at) {
        if constexpr (UA) return load_half8_any(base + min(at, last));
        const half8_t* src = reinterpret_cast<const half8_t*>(base + at);
        return NTL ? __builtin_nontemporal_load(src) : *src;
    };
    if (UA && coltile_nearly_full<RPP, R>(n)) {
        const uint32_t col = (uint32_t)(col0 < m ? col0 : col0 - (int32_t)(threadIdx.x % LPR) * 8);        // (past the row's end: the tile's first piece once more)
#pragma unroll
        for (int p = 0; p < R; ++p) v[p] = load((uint32_t)min(p * RPP + rg, n - 1) * (uint32_t)m + col);
    } else {
#pragma unroll
        for (int p = 0; p < R; ++p) v[p] = LOADS == kLoadsKept ? half8_kept(none) : half8_unset();
        uint32_t off = off0;
        asm volatile("" : "+v"(off));       // (or the addresses are kept in registers for coltile_store)
        if (col0 < m) {
#pragma unroll
            for (int p = 0; p < R; ++p)
                if (p * RPP + rg < n) v[p] = load(off + p * stride);
        }
    }
}

template <int NT, int LPR, int R, bool UA = false, int LOADS = coltile_loads(UA, R, LPR)>
__device__ inline void coltile_settle(half8_t (&v)[R], int32_t n, int32_t m, int32_t col0, half_t fill) {
    constexpr int RPP = NT / LPR;
    if constexpr (!UA) return;       // (right as they came)
    const int rg = threadIdx.x / LPR;
    half8_t none;
#pragma unroll
    for (int e = 0; e < 8; ++e) none[e] = fill;
    if (LOADS == kLoadsUnset || coltile_nearly_full<RPP, R>(n) || n * m < 8) {
#pragma unroll
        for (int p = 0; p < R; ++p)
            if ((p + 1) * RPP > n && p * RPP + rg >= n) v[p] = none;
    }
    if (col0 + 8 > m) {        // the piece across the rows' ends (its first m % 8 columns), or one past them
        const uint4_t keep = half8_keep(m - col0);
        const uint32_t over0 = (uint32_t)(col0 + 8) - (uint32_t)(n - rg) * (uint32_t)m, stride = (uint32_t)RPP * (uint32_t)m;
#pragma unroll
        for (int p = 0; p < R; ++p) {
            if (p * RPP < n) {
                // (rows that end less than a piece before the matrix does: the last one, several of less than a piece)
                const int32_t over = (int32_t)(over0 + p * stride);
                if ((p + 1) * RPP + 8 > n && p * RPP + rg < n && over > 0) v[p] = half8_down(v[p], over);
                v[p] = half8_fill(v[p], keep, none);
            }
        }
    }
}

template <int NT, int LPR, int R, bool NTL = false, bool UA = false, int LOADS = coltile_loads(UA, R, LPR)>
__device__ inline void coltile_load(half8_t (&v)[R], const half_t* base, int32_t n, int32_t m, int32_t col0, half_t fill) {
    coltile_request<NT, LPR, R, NTL, UA, LOADS>(v, base, n, m, col0, fill);
    coltile_settle<NT, LPR, R, UA, LOADS>(v, n, m, col0, fill);
}

template <int NT, int LPR, int R, bool NTS = false, bool UA = false>
__device__ inline void coltile_store(const half8_t (&v)[R], half_t* base, int32_t n, int32_t m, int32_t col0) {
    constexpr int RPP = NT / LPR;
    const int rg = threadIdx.x / LPR;
    const uint32_t off0 = (uint32_t)rg * (uint32_t)m + (uint32_t)col0, stride = (uint32_t)RPP * (uint32_t)m;
    if constexpr (UA) {
        if (col0 + 8 <= m) {
#pragma unroll
            for (int p = 0; p < R; ++p)
                if (p * RPP + rg < n) store_half8_any(base + (off0 + p * stride), v[p]);
        } else if (col0 < m) {
#pragma unroll
            for (int p = 0; p < R; ++p)
                if (p * RPP + rg < n) store_half8_head_any(base + (off0 + p * stride), m & 7, v[p]);
        }
    } else {
#pragma unroll
        for (int p = 0; p < R; ++p) {
            const int32_t row = p * RPP + rg;
            if (row < n && col0 < m) {
                half8_t* dst = reinterpret_cast<half8_t*>(base + (off0 + p * stride));
                if (NTS) __builtin_nontemporal_store(v[p], dst);
                else *dst = v[p];
            }
        }
    }
}

// v combined (sum or maximum) over the eight lanes of a wave that share lane % 8 -- lanes l, l ^ 8, l ^ 16, l ^ 32
// in that order, as three rounds of __shfl_xor would -- without the trips through the LDS crossbar: a rotation by
// 8 within each row of 16 lanes as an operand modifier, then the two lane-swap instructions of this architecture
// (v_permlane16_swap: odd rows of one register against even rows of the other; v_permlane32_swap: the halves).
template <bool IS_MAX>
__device__ __forceinline__ float lanes_mod8_combine(float v) {
    auto op = [](float a, float b) __attribute__((always_inline)) { return IS_MAX ? fmaxf(a, b) : a + b; };
    const uint32_t b0 = __builtin_bit_cast(uint32_t, v);
    v = op(v, __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b0, 0x128, 0xf, 0xf, true)));      // row_ror:8
    const uint32_t b1 = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(b1, b1, false, false);
    v = op(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
    const uint32_t b2 = __builtin_bit_cast(uint32_t, v);
    const auto q = __builtin_amdgcn_permlane32_swap(b2, b2, false, false);
    return op(__builtin_bit_cast(float, (uint32_t)q[0]), __builtin_bit_cast(float, (uint32_t)q[1]));
}

// The same for maxima of eight unsigned 16-bit numbers, two to a register.
__device__ __forceinline__ ushort8_t lanes_mod8_max(ushort8_t v) {
    uint4_t b = __builtin_bit_cast(uint4_t, v);
    typedef uint16_t ushort2_t __attribute__((ext_vector_type(2)));
    auto op = [](uint32_t x, uint32_t y) __attribute__((always_inline)) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(ushort2_t, x), __builtin_bit_cast(ushort2_t, y)));
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t x = b[i];
        x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, true));      // row_ror:8
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        x = op(r[0], r[1]);
        const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        b[i] = op(q[0], q[1]);
    }
    return __builtin_bit_cast(ushort8_t, b);
}

// Reduce NV groups of 8 per-lane column partials over all rows of the tile.  On return every
// lane holds the totals of its own 8 columns.  `lds` must hold (NT/64 + 1) * LPR*8 * NV floats.
template <int NT, int LPR, int NV, bool IS_MAX>
__device__ inline void coltile_reduce(float (&v)[NV * 8], float* lds) {
    constexpr int NW = NT / 64, COLS = LPR * 8, W = COLS * NV;
    if constexpr (LPR == 8 && !IS_MAX) {        // (for fp32 maxima the lane-swap form measured 4 % slower than the shuffles; those of halves go two to a register, lanes_mod8_max)
#pragma unroll
        for (int e = 0; e < NV * 8; ++e) v[e] = lanes_mod8_combine<IS_MAX>(v[e]);
    } else {
#pragma unroll
        for (int o = LPR; o < 64; o <<= 1) {
#pragma unroll
            for (int e = 0; e < NV * 8; ++e) {
                const float t = __shfl_xor(v[e], o, kWave);
                v[e] = IS_MAX ? fmaxf(v[e], t) : v[e] + t;
            }
        }
    }
    if (NW == 1) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (lane < LPR) {
#pragma unroll
        for (int g = 0; g < NV; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) lds[w * W + g * COLS + lane * 8 + e] = v[g * 8 + e];
    }
    __syncthreads();
    if (tid < W) {
        float r = lds[tid];
#pragma unroll
        for (int i = 1; i < NW; ++i) r = IS_MAX ? fmaxf(r, lds[i * W + tid]) : r + lds[i * W + tid];
        lds[NW * W + tid] = r;
    }
    __syncthreads();
    const int cg = tid % LPR;
#pragma unroll
    for (int g = 0; g < NV; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[g * 8 + e] = lds[NW * W + g * COLS + cg * 8 + e];
    __syncthreads();
}

// The same reduction for kernels that only hand the totals on (to their team): thread i < COLS*NV
// calls sink(i, total of packet i) -- packet g*COLS + c is statistic g of tile column c -- and
// nothing is read back, which saves two barriers.  Needs more than one wave.
template <int NT, int LPR, int NV, bool IS_MAX, class F>
__device__ inline void coltile_reduce_to(float (&v)[NV * 8], float* lds, F&& sink) {
    constexpr int NW = NT / 64, COLS = LPR * 8, W = COLS * NV;
    static_assert(NW > 1, "one wave has nothing to combine");
    if constexpr (LPR == 8 && !IS_MAX) {        // (for fp32 maxima the lane-swap form measured 4 % slower than the shuffles; those of halves go two to a register, lanes_mod8_max)
#pragma unroll
        for (int e = 0; e < NV * 8; ++e) v[e] = lanes_mod8_combine<IS_MAX>(v[e]);
    } else {
#pragma unroll
        for (int o = LPR; o < 64; o <<= 1) {
#pragma unroll
            for (int e = 0; e < NV * 8; ++e) {
                const float t = __shfl_xor(v[e], o, kWave);
                v[e] = IS_MAX ? fmaxf(v[e], t) : v[e] + t;
            }
        }
    }
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (lane < LPR) {
#pragma unroll
        for (int g = 0; g < NV; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) lds[w * W + g * COLS + lane * 8 + e] = v[g * 8 + e];
    }
    __syncthreads();
    if (tid < W) {
        float r = lds[tid];
#pragma unroll
        for (int i = 1; i < NW; ++i) r = IS_MAX ? fmaxf(r, lds[i * W + tid]) : r + lds[i * W + tid];
        sink(tid, r);
    }
}

}  // namespace cpmk
