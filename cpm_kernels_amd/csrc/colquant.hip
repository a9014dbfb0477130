// Per-column absmax scales and rounding of a (batch, n, m) fp16 tensor in one pass over HBM:
//   scale[b, j] = fp16(max_i |mat[b,i,j]| / 127),   q = int8(rint(mat[b,i,j] / scale[b,j]))
// i.e. cu_gemm_calc_scale_transpose followed by cu_gemm_round_transpose (cuda/gemm.cu:22-33,
// 79-98), with q written either in place (b, n, m) or transposed (b, m, n).  The transposed form
// is what lets torch-level bmm feed operands given as (batch, K, N) to the K-major int8 GEMM
// (the reference's GEMMInt8.forward, torch/gemm.py:84-113, quantises such an operand along
// dim 1 and leaves the transposition to cuBLASLt).  Or both: a product that will be differentiated
// needs the transposed form now and the other one for its backward pass.
// With row scales the values are mat[b,i,j] * row_scale[b,i] and the divisor is the fp32 absmax / 127
// (cu_gemm_backward_scale_round, cuda/gemm.cu:139-172): the gradient on its way to the product with
// the other operand.
// Either output may have rows longer than the matrix's, filled up with zeros: a product contracts over
// whole slabs then, whatever the number of rows or columns is.
#include "dim1.h"
#include "exchange.h"
#include "round_scale.h"

namespace cpmk {

// 64 columns x 512 rows per workgroup; taller columns are shared by a team (exchange.h) that
// exchanges the per-column maxima.  Lane (cg = tid % 8, rg = tid / 8) holds 8 columns of the 8
// consecutive rows rg*8 .. rg*8+7, so that its int8 results are 8 contiguous bytes in either
// output layout.
// Bound by the two memory phases of a workgroup -- all of its reads, then all of its writes -- around the wait for its team: without one
// (128 x 512 x 1024) it runs at 5.3 TB/s, with one at 4.0.  Three workgroups a compute unit (at most 80 registers per lane) while some
// wait: 8 x 10240 x 512 transposed 43.4 -> 37.1 us, with both outputs 48.4 -> 45.2, with row scales 51.5 -> 44.7; 16 x 4096 x 1024 57 -> 49.8;
// 8 x 4096 x 512, one round of the device, 19.2 -> 17.6.  Two a compute unit: 39.4, 46.8, 47.3, 52.7, 17.7; four (64 registers): 39.3, 50.3, 44.1, 50.9, 18.2.
// NTH: the tile's 128-byte row segments are whole cache lines (m % 64 == 0, the matrix on a 128-byte boundary): the input is
// read with the non-temporal hint.  Elsewhere a line is shared with the neighbouring tile and has to stay in L2 for it.
// UA: any m and alignment: a piece inside its row still moves whole, at whatever address it lies (global accesses need
// no alignment); the piece across a row's end is read with what lies behind it (and its scales and, not transposed, its int8 values are
// written) in at most three narrower accesses.
// OUT: bit 0 the transposed output, bit 1 the one in place.
struct ColQuantArgs {
    int32_t n, m;
    const half_t* mat;
    const half_t* row_scale;      // SCALED: (batch, n), or (n) shared by the batch
    int bc;
    half_t* scale;                // (batch, m)
    int8_t* out_t;                // (batch, m, ld_t)
    int8_t* out_n;                // (batch, n, ld_n)
    int32_t ld_t, ld_n;
};
constexpr int kOutT = 1, kOutN = 2;
// Parts of a team: the packets of all of them are dealt to the waves of a workgroup once, kColPackets to a wave.
constexpr int kColThreads = 512, kColPackets = 4;
constexpr int64_t kColMaxParts = kColThreads / 64 * kColPackets;

template <int NT, int OUT, bool NTH, bool UA, bool SCALED>
__device__ __forceinline__ void col_quantize_team(const ColQuantArgs& a, int32_t tiles_per_batch, int32_t parts, uint32_t nteams, const XchLaunch& xl) {
    constexpr bool TRANSPOSED = (OUT & kOutT) != 0, NATURAL = (OUT & kOutN) != 0;
    const int32_t n = a.n, m = a.m;
    const half_t* const mat = a.mat;
    half_t* const scale = a.scale;
    constexpr int LPR = 8, R = 8, COLS = 64, ROWS = NT / LPR * R;
    uint64_t* const xch = xl.region;
    const uint32_t tag = xl.tag;
    __shared__ __attribute__((aligned(16))) union { float f[NT / 64 * COLS]; uint16_t h[NT / 64 * COLS]; } wmax;       // column maxima of each wave
    __shared__ float xmax[NT];                                    // the team's column maxima, [wave][column]
    __shared__ __attribute__((aligned(16))) float colscale[COLS], colrcp[COLS];
    __shared__ bool all_normal;
    __shared__ __attribute__((aligned(16))) int8_t tbuf[TRANSPOSED ? COLS * ROWS : 16];       // the transposed int8 tile on its way out
    const int tid = threadIdx.x, cg = tid % LPR, rg = tid / LPR;
    XchMember me;
    if (!xch_member(blockIdx.x, parts, nteams, me)) return;
    const uint32_t part = me.part, team = me.team;
    const uint32_t b = team / tiles_per_batch, ct = team - b * tiles_per_batch;
    const int32_t col0 = ct * COLS + cg * 8;
    const int32_t row0 = part * ROWS + rg * 8;           // this lane's first row
    const int64_t boff = (int64_t)b * n * m;

    half_t sxh[SCALED ? R : 1];        // the lane's rows' scales, requested ahead of the tile (each under a condition they waited for one another)
    if constexpr (SCALED) {
        const half_t* rs = a.row_scale + (a.bc ? 0 : (int64_t)b * n);
#pragma unroll
        for (int p = 0; p < R; ++p) sxh[p] = rs[min(row0 + p, n - 1)];
    }
    // one lane offset beside a scalar address per row of the lane (n * m < 2^31: the offset in bytes of a row within the matrix fits)
    const half_t* const tbase = mat + boff + (int64_t)part * ROWS * m;
    const uint32_t loff = ((uint32_t)(rg * 8) * (uint32_t)m + (uint32_t)col0) * 2u;
    half8_t v[R];
    const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const bool narrow = UA && (int64_t)n * m < 8;        // (a matrix of less than a piece)
    if (UA && !narrow) {
        // Every load is made, rows past the last as the last one, and put right behind them all; waves that have no rows leave them out
        const half_t* const mb = mat + boff;
        const uint32_t last = (uint32_t)n * (uint32_t)m - 8u, col = (uint32_t)min(col0, m - 1);
        if (!(SCALED && NATURAL) && __builtin_amdgcn_readfirstlane(row0) >= n) {        // (80 registers do not hold that choice beside the scales and the outputs in place)
#pragma unroll
            for (int p = 0; p < R; ++p) v[p] = zero8;
        } else {
#pragma unroll
            for (int p = 0; p < R; ++p) v[p] = load_half8_any(mb + min((uint32_t)min(row0 + p, n - 1) * (uint32_t)m + col, last));
            if (col0 + 8 > m && row0 < n) {
                const uint4_t keep = half8_keep(m - col0);
                const uint32_t over0 = (uint32_t)(col0 + 8) - (uint32_t)(n - row0) * (uint32_t)m;       // (rows that end less than a piece before the matrix's end: the last one, several of less than a piece)
#pragma unroll
                for (int p = 0; p < R; ++p) {
                    const int32_t over = (int32_t)(over0 + (uint32_t)p * (uint32_t)m);
                    if (over > 0 && over < 8) v[p] = half8_down(v[p], over);
                    v[p] = half8_fill(v[p], keep, zero8);
                }
            }
            if (row0 + R > n) {
#pragma unroll
                for (int p = 0; p < R; ++p)
                    if (row0 + p >= n) v[p] = zero8;
            }
        }
    } else {
#pragma unroll
        for (int p = 0; p < R; ++p) {
            v[p] = zero8;
            const half_t* const src = reinterpret_cast<const half_t*>(reinterpret_cast<const char*>(tbase + (int64_t)p * m) + loff);
            if (row0 + p < n && col0 < m) {
                if constexpr (UA) {
                    v[p] = load_half8_head_any(src, m & 7, zero8);
                } else {
                    const half8_t* src8 = reinterpret_cast<const half8_t*>(src);
                    v[p] = NTH ? __builtin_nontemporal_load(src8) : *src8;        // read once; the int8 output below is what the next kernel wants in cache
                }
            }
        }
    }
    float sx[SCALED ? R : 1];
    if constexpr (SCALED) {
#pragma unroll
        for (int p = 0; p < R; ++p) sx[p] = row0 + p < n ? (float)sxh[p] : 0.0f;
    }
    // The maxima over the rows of a wave, then over the workgroup's waves: thread i < COLS ends up with that of column i.
    float M = 0.0f;
    if constexpr (SCALED) {
        float mx[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) mx[e] = 0.0f;
#pragma unroll
        for (int p = 0; p < R; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) mx[e] = fmaxf(mx[e], fabsf((float)v[p][e] * sx[p]));       // (skips NaN products, as the reference's fmaxf does)
        coltile_reduce_to<NT, LPR, 1, true>(mx, wmax.f, [&](int, float r) { M = r; });
    } else {
        // |x| of the lane's 8 columns as integers, two to a register all the way through; a NaN among them (rare) repeats the maximum in
        // floating point, which skips NaN elements
        ushort8_t um = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < R; ++p) um = absbits_max(um, v[p]);
        if (absbits_max_of(um) > 0x7c00u) {
            half8_t hm = __builtin_elementwise_abs(v[0]);
#pragma unroll
            for (int p = 1; p < R; ++p) hm = __builtin_elementwise_max(hm, __builtin_elementwise_abs(v[p]));
#pragma unroll
            for (int e = 0; e < 8; ++e) hm[e] = hm[e] != hm[e] ? (half_t)0.0f : hm[e];       // (nothing but NaN)
            um = __builtin_bit_cast(ushort8_t, hm);
        }
        um = lanes_mod8_max(um);
        if ((tid & 63) < LPR) *reinterpret_cast<ushort8_t*>(wmax.h + (tid >> 6) * COLS + cg * 8) = um;
        __syncthreads();
        if (tid < COLS) {
            uint16_t r = wmax.h[tid];
#pragma unroll
            for (int w = 1; w < NT / 64; ++w) r = max(r, wmax.h[w * COLS + tid]);
            M = (float)__builtin_bit_cast(half_t, r);
        }
    }
    if (parts > 1) {
        // The packets of the team's parts are dealt to the waves, four to a thread, which all wait at the same time: one wave asking for
        // eight at a time held 40 registers and went through them in turn.
        static_assert(NT / 64 * kColPackets >= kColMaxParts, "a part beyond these would be left out of the maxima");
        uint64_t* team_slots = xch + (size_t)team * parts * kXchVals;
        if (tid < COLS) xch_post(team_slots + (size_t)part * kXchVals, tid, M, tag);
        const int w = tid >> 6;
        static_assert(kColPackets == 4, "the maximum below");
        float x[kColPackets];
        const bool ok = xch_gather<kColPackets>(team_slots, parts, w * kColPackets, tid & 63, tag, wall_clock64() + kXchTimeoutTicks, x);
        const float m4 = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));       // maxima are >= 0: absent parts (zeros) do not matter
        xmax[tid] = ok ? m4 : __builtin_nanf("");
        if (!ok) xch_flag(xl, kXchStatusTimeout);
        __syncthreads();
    }
    // One wave: the maximum of each column, its scale and the reciprocal, for all lanes of the column (a lane's 16 divisions, if
    // each made its own eight columns', were a quarter of the kernel's instructions).
    if (tid < COLS) {
        if (parts > 1) {
            M = xmax[tid];
#pragma unroll
            for (int w = 1; w < NT / 64; ++w) {
                const float x = xmax[w * COLS + tid];
                M = x > M || x != x ? x : M;       // (a NaN, where a packet did not arrive, stays)
            }
        }
        // (columns past the matrix's edge get a scale of 1: theirs of 0 would send the whole tile through the long rounding sequence,
        // 32 x 359 with row scales 10.8 us, 8.9 so; 8 x 4096 x 500 25.9 -> 23.6)
        const int32_t col = ct * COLS + tid;
        if (col >= m) M = 127.0f;
        const float s1 = SCALED ? (float)((double)M / 127.0) : 0.0f;       // float / double constant, as the reference writes it
        const half_t sh = SCALED ? (half_t)s1 : scale_from_absmax(M);
        const float s = SCALED ? s1 : (float)sh;
        // A column of nothing but zeros and NaN (a padded token's, a masked gradient's) is 0 everywhere: the short sequence gives that with
        // a reciprocal of 0 too, and the 63 columns beside it stay on it (8 x 4096 x 512 with one such column a tile 25.5 -> 17.7 us).
        const bool empty = M == 0.0f;
        colscale[tid] = s;
        colrcp[tid] = empty ? 0.0f : 1.0f / s;
        const bool normal = empty || (SCALED ? own_scale_in_range(s) : scale_is_normal(sh));
        const bool every = __builtin_amdgcn_ballot_w64(!normal) == 0;
        if (tid == 0) all_normal = every;
        if (part == 0 && col < m) scale[(int64_t)b * m + col] = sh;
    }
    __syncthreads();

    uint32_t q[R][2];       // [row p][columns 0-3 | 4-7], one byte each
    if (all_normal) {    // every scale of the tile's columns is a normal number: the short rounding sequence
        float s[8], y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            y[e] = colrcp[cg * 8 + e];
            s[e] = SCALED ? colscale[cg * 8 + e] : 0.0f;
        }
#pragma unroll
        for (int p = 0; p < R; ++p) {
            uint32_t t[8];
            int4_t vp = __builtin_bit_cast(int4_t, v[p]);
            asm volatile("" : "+v"(vp));             // keeps the fp32 conversions of the two paths apart (hoisted above the branch they hold 64 registers)
            const half8_t vh = __builtin_bit_cast(half8_t, vp);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                t[e] = SCALED ? quant_i8_own_fp32_scale_bits((float)vh[e] * sx[p], s[e], y[e]) : quant_i8_own_scale_bits((float)vh[e], y[e]);
            q[p][0] = pack4_i8((int32_t)t[0], (int32_t)t[1], (int32_t)t[2], (int32_t)t[3]);
            q[p][1] = pack4_i8((int32_t)t[4], (int32_t)t[5], (int32_t)t[6], (int32_t)t[7]);
            __builtin_amdgcn_sched_barrier(0);      // one row at a time: interleaving all 64 elements costs registers
        }
    } else {
        // A scale below the normal numbers, or not finite.  Four columns at a time, so that scales and reciprocals are eight registers
        // (8 x 4096 x 512 with one such column a tile 25.7 -> 20.5 us, against one IEEE division an element, one element at a time).
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4_t s = *reinterpret_cast<const float4_t*>(colscale + cg * 8 + h * 4), y = *reinterpret_cast<const float4_t*>(colrcp + cg * 8 + h * 4);
#pragma unroll
            for (int p = 0; p < R; ++p) {
                int32_t t[4];
                int4_t vp = __builtin_bit_cast(int4_t, v[p]);
                asm volatile("" : "+v"(vp));             // (what was computed for the maxima is not to be kept for here)
                const half8_t vh = __builtin_bit_cast(half8_t, vp);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (SCALED) {
                        t[e] = quant_i8((float)vh[h * 4 + e] * sx[p], s[e]);
                        __builtin_amdgcn_sched_barrier(0);      // one division at a time: infinite products only, which are not to set the register count
                    } else {
                        t[e] = quant_i8_rcp((float)vh[h * 4 + e], s[e], y[e]);
                    }
                }
                q[p][h] = pack4_i8(t[0], t[1], t[2], t[3]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if constexpr (NATURAL) {
        if (col0 < a.ld_n) {
            int8_t* const obase = a.out_n + (int64_t)b * n * a.ld_n + (int64_t)part * ROWS * a.ld_n;
            const uint32_t ooff = (uint32_t)(rg * 8) * (uint32_t)a.ld_n + (uint32_t)col0;
#pragma unroll
            for (int p = 0; p < R; ++p)
                if (row0 + p < n) {
                    int8_t* dst = obase + (int64_t)p * a.ld_n + ooff;
                    if constexpr (UA) {       // (ld_n is m, or a multiple of 16 beyond it: the piece across the matrix's edge ends in zeros then)
                        if (col0 + 8 <= a.ld_n) store_byte8_any(dst, q[p][0], q[p][1]);
                        else store_byte8_head_any(dst, a.ld_n & 7, q[p][0], q[p][1]);
                    } else {
                        *reinterpret_cast<uint2_t*>(dst) = uint2_t{q[p][0], q[p][1]};
                    }
                }
        }
    }
    if constexpr (TRANSPOSED) {
        // The tile leaves through LDS as 64 columns x ROWS bytes: a lane's 8 rows of a column are 8
        // bytes there, and 32 lanes then store one column's ROWS bytes as one contiguous run (16 bytes
        // per lane) instead of eight lanes storing 64 bytes of it.  8-byte slot s of column c sits at
        // slot s ^ ((c / 8) * 8): the 64 lanes of a writing wave cover every bank equally, and the
        // 16-byte reads stay pairs of neighbouring slots.
        static_assert(ROWS == 512, "one column of the tile is 64 slots of 8 bytes");
        // 4x4 byte transposes with v_perm_b32 (selector bytes 0-3 pick from the second operand, 4-7 from
        // the first): tr[h][e4][k] = rows 4k .. 4k+3 of column 4h + e4
        uint32_t tr[2][4][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t r0 = q[4 * k][h], r1 = q[4 * k + 1][h], r2 = q[4 * k + 2][h], r3 = q[4 * k + 3][h];
                const uint32_t a01 = __builtin_amdgcn_perm(r1, r0, 0x05010400u), b01 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
                const uint32_t a23 = __builtin_amdgcn_perm(r3, r2, 0x05010400u), b23 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
                tr[h][0][k] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
                tr[h][1][k] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
                tr[h][2][k] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
                tr[h][3][k] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
            }
#pragma unroll
        for (int e = 0; e < 8; ++e)
            *reinterpret_cast<uint2_t*>(tbuf + (cg * 8 + e) * ROWS + ((rg ^ (cg << 3)) << 3)) = uint2_t{tr[e >> 2][e & 3][0], tr[e >> 2][e & 3][1]};
        __syncthreads();
        const int piece = tid & 31;                                  // 16 rows of a column
        const int32_t prow = part * ROWS + piece * 16;
#pragma unroll
        for (int ps = 0; ps < COLS / (NT / 32); ++ps) {
            const int c = ps * (NT / 32) + (tid >> 5);
            const int32_t col = ct * COLS + c;
            const int4_t w = *reinterpret_cast<const int4_t*>(tbuf + c * ROWS + (((piece * 2) ^ ((c >> 3) << 3)) << 3));
            int8_t* dst = a.out_t + (int64_t)b * m * a.ld_t + ((uint32_t)col * (uint32_t)a.ld_t + (uint32_t)prow);
            if (col < m) {             // ld_t % 8 == 0: a piece is whole, half or not there
                if (prow + 16 <= a.ld_t) *reinterpret_cast<int4_t*>(dst) = w;
                else if (prow + 8 <= a.ld_t) *reinterpret_cast<uint2_t*>(dst) = uint2_t{(uint32_t)w.x, (uint32_t)w.y};
            }
        }
    }
    if (parts > 1 && tid < 64) xch_retire(xl, team, parts);
}

template <int NT, int OUT, bool NTH, bool UA, bool SCALED>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(6, 6))) void k_col_quantize_team(ColQuantArgs a, int32_t tiles_per_batch, int32_t parts,
                                                          uint32_t nteams, XchLaunch xl) {
    col_quantize_team<NT, OUT, NTH, UA, SCALED>(a, tiles_per_batch, parts, nteams, xl);
}

// The other operand of the same product, quantised along its rows, in the same launch (k_col_quantize_rows): its workgroups follow the
// teams', and stream while those wait for their members and for their phases to pass.  Bound by memory: an 8 x 4096 x 512 and an 8 x 10240 x 512
// operand beside their 10240 x 4096 weights, 428 MB, 82 us (5.2 TB/s) where a launch for each takes 90; 4 x 2944 x 296 beside 2944 rows 15 and 18,
// 2 x 1024 x 72 beside 824 9 and 12.  Six waves a SIMD for the rows too, as for the teams; a wave a row up to 4096 columns, a workgroup beyond.
struct RowQuantArgs {
    const half_t* mat;            // (rows, m), m % 8 == 0, 16-byte aligned
    half_t* scale;
    int8_t* out;                  // (rows, ld), 8-byte aligned, ld % 8 == 0: the surplus is zeros
    int32_t m, ld;
    int64_t rows;
    uint32_t first;               // number of the first workgroup of the rows
};

// A row's pieces of eight, NV of them a lane, `step` pieces apart; ROW_WG: the row is the whole workgroup's, else a wave's.
template <int NV, bool ROW_WG>
__device__ __forceinline__ void quantize_row(const RowQuantArgs& a, uint32_t block) {
    __shared__ uint32_t red[kColThreads / 64];
    __shared__ float redf[kColThreads / 64];
    constexpr int STEP = ROW_WG ? kColThreads : 64;
    const int tid = threadIdx.x, lane = ROW_WG ? tid : tid & 63;
    const int64_t row = ROW_WG ? (int64_t)block : (int64_t)block * (kColThreads / 64) + (tid >> 6);
    if (row >= a.rows) return;                        // (the same for the whole workgroup where it meets at barriers)
    const half8_t* p8 = reinterpret_cast<const half8_t*>(a.mat + row * a.m);
    const int m8 = a.m >> 3, l8 = a.ld >> 3;
    half8_t v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        v[i] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
        if (lane + i * STEP < m8) v[i] = __builtin_nontemporal_load(p8 + lane + i * STEP);
    }
    ushort8_t um = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NV; ++i) um = absbits_max(um, v[i]);
    uint32_t ub = wave_max_u32_uniform(absbits_max_of(um));
    if constexpr (ROW_WG) {
        if ((tid & 63) == 0) red[tid >> 6] = ub;
        __syncthreads();
        ub = red[0];
#pragma unroll
        for (int w = 1; w < kColThreads / 64; ++w) ub = max(ub, red[w]);
    }
    float mx = (float)__builtin_bit_cast(half_t, (uint16_t)ub);
    if (ub > 0x7c00u) {      // (the same for the whole row) a NaN: the maximum that skips NaN elements
        mx = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            int4_t ci = __builtin_bit_cast(int4_t, v[i]);
            asm volatile("" : "+v"(ci));         // nothing of this rare path is to be computed ahead of the branch
            const half8_t h = __builtin_bit_cast(half8_t, ci);
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(fabsf((float)h[e]), mx);
        }
        if constexpr (ROW_WG) mx = block_max<kColThreads / 64>(mx, redf);
        else mx = wave_max(mx);
    }
    const half_t sh = scale_from_absmax(mx);
    if (lane == 0) a.scale[row] = sh;
    const float s = (float)sh, y = 1.0f / s;
    uint2_t* const orow = reinterpret_cast<uint2_t*>(a.out + row * a.ld);
    const bool normal = scale_is_normal(sh);       // (the same for the whole row) the short rounding sequence
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = lane + i * STEP;
        int4_t ci = __builtin_bit_cast(int4_t, v[i]);
        asm volatile("" : "+v"(ci));             // (a piece's fp32 conversions are made where they are used)
        const half8_t h = __builtin_bit_cast(half8_t, ci);
        int32_t q[8];
        if (normal) {
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] = (int32_t)quant_i8_own_scale_bits((float)h[e], y);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] = quant_i8_rcp((float)h[e], s, y);
        }
        if (j < l8) orow[j] = uint2_t{pack4_i8(q[0], q[1], q[2], q[3]), pack4_i8(q[4], q[5], q[6], q[7])};
    }
}

template <int OUT, bool NTH, bool UA>
__global__ __launch_bounds__(kColThreads) __attribute__((amdgpu_waves_per_eu(6, 6))) void k_col_quantize_rows(ColQuantArgs a, int32_t tiles_per_batch, int32_t parts,
                                                                                                            uint32_t nteams, XchLaunch xl, RowQuantArgs r) {
    if (blockIdx.x < r.first) {
        col_quantize_team<kColThreads, OUT, NTH, UA, false>(a, tiles_per_batch, parts, nteams, xl);
        return;
    }
    const uint32_t block = blockIdx.x - r.first;
    const int32_t len = r.ld;                    // (ld >= m)
    if (len <= 1024) quantize_row<2, false>(r, block);
    else if (len <= 2048) quantize_row<4, false>(r, block);
    else if (len <= 4096) quantize_row<8, false>(r, block);
    else if (len <= 8192) quantize_row<2, true>(r, block);
    else if (len <= 12288) quantize_row<3, true>(r, block);
    else quantize_row<4, true>(r, block);
}

// The gradient on its way to both products of a backward pass: its columns and its rows in one launch, as above, bound the same way; rows that a wave holds in
// registers (75 of them beside the teams' 80, no LDS).  A launch for each / one, operands outside the caches, us: 8 x 10240 x 512 84 / 79, 8 x 4096 x 512 41.4 / 35.7, 4 x 10240 x 500
// 66 / 50, 15 x 2048 x 736 52 / 46, 4 x 896 x 172 27 / 19.5, 16 x 4096 x 1024 112 / 112.
template <bool NTH, bool UA>
__global__ __launch_bounds__(kColThreads) __attribute__((amdgpu_waves_per_eu(6, 6))) void k_col_scale_round_rows(ColQuantArgs a, int32_t tiles_per_batch, int32_t parts,
                                                                                                               uint32_t nteams, XchLaunch xl, RoundScaleArgs r) {
    if (blockIdx.x < r.first) {
        col_quantize_team<kColThreads, kOutT, NTH, UA, true>(a, tiles_per_batch, parts, nteams, xl);
        return;
    }
    const int64_t wave = (int64_t)(blockIdx.x - r.first) * (kColThreads / 64) + (threadIdx.x >> 6);
    if (r.m <= 512) round_scale_rows_reg<1, 4, UA, true>(r, wave);
    else if (r.m <= 1024) round_scale_rows_reg<2, 2, UA, true>(r, wave);
    else round_scale_rows_reg<4, 1, UA, true>(r, wave);
}

// Rows r0 .. r0 + 63 of a tile of 64 columns, rounded with the scale of the lane's column, into the wanted outputs (256 threads;
// the transposed one through `tile`, so that a wave stores 64 bytes of one column and not one of 64).  The surplus of longer
// rows becomes zeros: rows from n on in the transposed output, columns from m on in the other.
__device__ __forceinline__ void col_round_tile(const ColQuantArgs& a, int64_t b, int32_t col0, int32_t r0, float s, int8_t (&tile)[64][68]) {
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const int32_t n = a.n, m = a.m, col = col0 + c;
    const half_t* mat = a.mat + b * n * m;
    const half_t* rs = a.row_scale ? a.row_scale + (a.bc ? 0 : b * n) : nullptr;
    float x[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const int32_t i = r0 + p * 4 + rg;
        x[p] = col < m && i < n ? (float)mat[(int64_t)i * m + col] * (rs ? (float)rs[i] : 1.0f) : 0.0f;
    }
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const int32_t i = r0 + p * 4 + rg;
        const int8_t q = col < m && i < n ? (int8_t)quant_i8(x[p], s) : 0;
        tile[c][p * 4 + rg] = q;
        if (a.out_n && col < a.ld_n && i < n) a.out_n[(b * n + i) * a.ld_n + col] = q;
    }
    if (a.out_t == nullptr) return;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const int32_t j = col0 + p * 4 + rg;
        if (j < m && r0 + c < a.ld_t) a.out_t[(b * m + j) * a.ld_t + r0 + c] = tile[p * 4 + rg][c];
    }
}

// Any shape, columns taller than a team holds or launches recorded when no packets are left: the rounding with scales that
// are there already, 64 x 64 elements per workgroup.
__global__ __launch_bounds__(256) void k_col_round_any(ColQuantArgs a, int32_t col_tiles, int32_t rt0) {
    __shared__ int8_t tile[64][68];
    const uint32_t rt = blockIdx.x / (uint32_t)col_tiles;
    const int32_t col0 = (int32_t)(blockIdx.x - rt * (uint32_t)col_tiles) * 64;
    const int64_t b = blockIdx.y;
    const int32_t col = col0 + (threadIdx.x & 63);
    col_round_tile(a, b, col0, (rt0 + (int32_t)rt) * 64, col < a.m ? (float)a.scale[b * a.m + col] : 1.0f, tile);
}

// The same shapes with row scales, where the divisor is the fp32 absmax / 127 and not the fp16 scale that is kept: both passes in
// one workgroup per 64 columns.
__global__ __launch_bounds__(256) void k_col_scale_round_any(ColQuantArgs a) {
    __shared__ float red[4][64];
    __shared__ int8_t tile[64][68];
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const int32_t n = a.n, m = a.m, col0 = blockIdx.x * 64, col = col0 + c;
    const int64_t b = blockIdx.y;
    const half_t* mat = a.mat + b * n * m;
    const half_t* rs = a.row_scale + (a.bc ? 0 : b * n);
    float mx = 0.0f;
    if (col < m) {
#pragma unroll 8
        for (int32_t i = rg; i < n; i += 4) mx = fmaxf(mx, fabsf((float)mat[(int64_t)i * m + col] * (float)rs[i]));
    }
    red[rg][c] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0][c], red[1][c]), fmaxf(red[2][c], red[3][c]));
    const float s = (float)((double)mx / 127.0);
    if (rg == 0 && col < m) a.scale[b * m + col] = (half_t)s;
    for (int32_t r0 = 0; r0 < max(n, a.ld_t); r0 += 64) {
        col_round_tile(a, b, col0, r0, s, tile);
        __syncthreads();       // (the tile has left before the next one)
    }
}

// Any shape: rounding with per-column scales into the transposed layout, one element per thread.
__global__ __launch_bounds__(256) void k_round_cols_transposed(int64_t total, int32_t n, int32_t m,
                                                               const half_t* __restrict__ mat,
                                                               const half_t* __restrict__ scale,
                                                               int8_t* __restrict__ out) {
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= total) return;
    const int64_t bi = gid / m;                 // b*n + i
    const int32_t j = (int32_t)(gid - bi * m);
    const int64_t b = bi / n;
    const int32_t i = (int32_t)(bi - b * n);
    out[(b * m + j) * n + i] = (int8_t)quant_i8((float)mat[gid], (float)scale[b * m + j]);
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_gemm_calc_scale_transpose(int32_t, int32_t, int32_t, const void*, void*, void*);
int cpmk_gemm_round_transpose(int32_t, int32_t, int32_t, const void*, const void*, void*, void*);

}  // extern "C"

// The team kernel on (batch, n, m): 0, an error code, or -1 when the shape is not one it takes.  rq: rows to quantise beside the (first)
// launch of the teams; -1 also where they are not of the form that takes.
template <bool SCALED>
static int col_quantize(int32_t batch, const ColQuantArgs& p, hipStream_t st, const std::conditional_t<SCALED, RoundScaleArgs, RowQuantArgs>* rq = nullptr) {
    const int32_t n = p.n, m = p.m;
    // a team here exchanges one maximum per column, dealt to all waves, so it may be larger than the teams of the kernels that keep
    // per-part values in registers (kColMaxParts of 512 rows: 16384; far fewer workgroups than are resident at once, which is what progress
    // needs)
    const int64_t tiles = ceil_div(p.out_n ? p.ld_n : m, 64), parts = ceil_div(n, 512);
    // rows of whole 16-byte pieces in aligned buffers: 16-byte accesses; any other width or alignment: the same kernel moving
    // its columns one by one (the transposed output runs along n either way)
    const bool wide = (m % 8 == 0) && aligned16(p.mat) && aligned16(p.scale) && ((reinterpret_cast<uintptr_t>(p.out_n) & 7u) == 0);
    const bool team_ok = (!p.out_t || (p.ld_t % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out_t) & 7u) == 0)) &&
                         (int64_t)n * (p.out_n ? p.ld_n : m) < (1ll << 31) && (int64_t)m * p.ld_t < (1ll << 31) && p.ld_t <= parts * 512 &&
                         parts <= kColMaxParts && tiles * parts <= kXchSlots;
    if (!team_ok) return -1;
    int64_t row_blocks = 0;
    if (rq) {
        if constexpr (SCALED) {
            row_blocks = ceil_div(rq->rows, kColThreads / 64 * (rq->m <= 512 ? 4 : rq->m <= 1024 ? 2 : 1));
            if (rq->m > 2048 || (wide && (!aligned16(rq->scale_y) || (reinterpret_cast<uintptr_t>(rq->out) & 7u)))) return -1;
        } else {
            row_blocks = rq->ld > 4096 ? rq->rows : ceil_div(rq->rows, kColThreads / 64);
            if (rq->m % 8 || rq->ld % 8 || rq->ld > 16384 || !aligned16(rq->mat) || (reinterpret_cast<uintptr_t>(rq->out) & 7u)) return -1;
        }
        if (row_blocks > 1 << 21) return -1;
    }
    // teams use one packet slot per (team, part): batches beyond the pool go out in several launches
    const int64_t per_launch = parts > 1 ? kXchSlots / (tiles * parts) : ((1ll << 31) - 8) / (tiles * parts);
    for (int64_t b0 = 0; b0 < batch; b0 += per_launch) {
        const int64_t nb = batch - b0 < per_launch ? batch - b0 : per_launch;
        XchScope xs;
        if (parts > 1) {
            const int rc = xs.begin(tiles * nb * parts, st);
            if (rc == kXchFull && b0 == 0) return -1;       // recorded into a graph and the capture reserve is used up: the separate kernels
            if (rc != 0) return rc == kXchFull ? CPMK_ETOOBIG : rc;
        }
        const bool lines = m % 64 == 0 && (reinterpret_cast<uintptr_t>(p.mat) & 127u) == 0;
        ColQuantArgs q = p;
        q.mat += b0 * n * m;
        if (p.row_scale && !p.bc) q.row_scale += b0 * n;
        q.scale += b0 * m;
        if (p.out_t) q.out_t += b0 * m * p.ld_t;
        if (p.out_n) q.out_n += b0 * n * p.ld_n;
        const int64_t team_blocks = xch_team_grid(tiles * nb, parts);
        auto go_rows = [&](auto kern) {
            auto r = *rq;
            r.first = (uint32_t)team_blocks;
            hipLaunchKernelGGL(kern, dim3((unsigned)(team_blocks + row_blocks)), dim3(kColThreads), 0, st, q, (int32_t)tiles, (int32_t)parts, (uint32_t)(tiles * nb),
                               xs.xl, r);
        };
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((unsigned)team_blocks), dim3(kColThreads), 0, st, q, (int32_t)tiles, (int32_t)parts,
                               (uint32_t)(tiles * nb), xs.xl);
        };
        auto pick = [&](auto oc) {
            constexpr int OUT = decltype(oc)::value;
            if constexpr (!SCALED && (OUT & kOutT) != 0) {
                if (rq && b0 == 0) {
                    if (!wide) go_rows(k_col_quantize_rows<OUT, false, true>);
                    else if (lines) go_rows(k_col_quantize_rows<OUT, true, false>);
                    else go_rows(k_col_quantize_rows<OUT, false, false>);
                    return;
                }
            }
            if constexpr (SCALED) {
                if (rq && b0 == 0) {        // (rows beside columns: the transposed output only)
                    if (!wide) go_rows(k_col_scale_round_rows<false, true>);
                    else if (lines) go_rows(k_col_scale_round_rows<true, false>);
                    else go_rows(k_col_scale_round_rows<false, false>);
                    return;
                }
            }
            if (!wide) go(k_col_quantize_team<kColThreads, OUT, false, true, SCALED>);
            else if (lines) go(k_col_quantize_team<kColThreads, OUT, true, false, SCALED>);
            else go(k_col_quantize_team<kColThreads, OUT, false, false, SCALED>);
        };
        if (p.out_t && p.out_n) {
            if constexpr (!SCALED) pick(std::integral_constant<int, kOutT | kOutN>{});
        } else if (p.out_t) {
            pick(std::integral_constant<int, kOutT>{});
        } else {
            pick(std::integral_constant<int, kOutN>{});
        }
        const int e = launch_status();
        const int rc2 = xs.end();
        if (e != 0 || rc2 != 0) return e ? e : rc2;
    }
    return 0;
}

namespace cpmk {
int col_scale_round_team(int32_t batch, int32_t n, int32_t m, const void* mat, const void* row_scale, int bc, void* scale, void* out, void* stream) {
    const ColQuantArgs p = {n, m, (const half_t*)mat, (const half_t*)row_scale, bc, (half_t*)scale, nullptr, (int8_t*)out, 0, m};
    return col_quantize<true>(batch, p, (hipStream_t)stream);
}
}  // namespace cpmk

extern "C" {

int cpmk_gemm_quantize_cols(int32_t batch, int32_t n, int32_t m, const void* mat, void* scale, void* out,
                            int out_transposed, void* stream) {
    clear_stale_error();
    if (batch < 0 || n < 0 || m < 0) return CPMK_EBADARG;
    if ((int64_t)batch * m == 0) return 0;
    if (n == 0) return cpmk_gemm_calc_scale_transpose(batch, n, m, mat, scale, stream);       // (columns of no elements: scale 0, nothing to round)
    if (any_null(mat, scale, out)) return CPMK_EBADARG;
    hipStream_t st = (hipStream_t)stream;
    const ColQuantArgs p = {n, m, (const half_t*)mat, nullptr, 0, (half_t*)scale, out_transposed ? (int8_t*)out : nullptr,
                            out_transposed ? nullptr : (int8_t*)out, out_transposed ? n : 0, out_transposed ? 0 : m};
    const int rc = col_quantize<false>(batch, p, st);
    if (rc >= 0) return rc;
    if (int e = cpmk_gemm_calc_scale_transpose(batch, n, m, mat, scale, stream)) return e;
    if (!out_transposed) return cpmk_gemm_round_transpose(batch, n, m, mat, scale, out, stream);
    const int64_t total = (int64_t)batch * n * m;
    hipLaunchKernelGGL(k_round_cols_transposed, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, total, n, m,
                       (const half_t*)mat, (const half_t*)scale, (int8_t*)out);
    return launch_status();
}

int cpmk_gemm_quantize_cols_ld(int32_t batch, int32_t n, int32_t m, const void* mat, const void* row_scale, int broad_cast_row,
                               void* scale, void* out_t, int32_t ld_t, void* out_n, int32_t ld_n, void* stream) {
    clear_stale_error();
    if (batch < 0 || n < 0 || m < 0 || (out_t && (ld_t < n || ld_t % 16)) || (out_n && (ld_n < m || (ld_n != m && ld_n % 16)))) return CPMK_EBADARG;
    if ((int64_t)batch * m == 0) return 0;       // (before the buffers are looked at: those of an empty problem may be null)
    if (scale == nullptr) return CPMK_EBADARG;
    if (n > 0) {       // (columns of no elements: scale 0 and whatever lengthens their rows)
        if ((out_t == nullptr) == (out_n == nullptr) && (row_scale || out_t == nullptr)) return CPMK_EBADARG;       // (both outputs: without row scales only)
        if (mat == nullptr) return CPMK_EBADARG;
    }
    const ColQuantArgs p = {n, m, (const half_t*)mat, (const half_t*)row_scale, broad_cast_row, (half_t*)scale, (int8_t*)out_t, (int8_t*)out_n,
                            out_t ? ld_t : 0, out_n ? ld_n : 0};
    const int rc = n == 0 ? -1 : row_scale ? col_quantize<true>(batch, p, (hipStream_t)stream) : col_quantize<false>(batch, p, (hipStream_t)stream);
    if (rc >= 0) return rc;
    // Scales by a workgroup per 64 columns, then the rounding by tiles over the whole device: a product of 512 rows and (20480, 4096)
    // quantised along 20480 takes 406 us, 4051 with both in one kernel that stored the transposed values byte by byte.  Row scales
    // need the fp32 divisor, which is not kept: one kernel, transposed through LDS (the gradient of such an operand 4.9 -> 2.7 ms).
    if (row_scale == nullptr)
        if (int e = cpmk_gemm_calc_scale_transpose(batch, n, m, mat, scale, stream)) return e;
    const int64_t col_tiles = ceil_div(p.out_n ? p.ld_n : m, 64), row_tiles = ceil_div(n > p.ld_t ? n : p.ld_t, 64);
    const int64_t per_launch = (1 << 23) / col_tiles > 0 ? (1 << 23) / col_tiles : 1;       // row tiles (a launch holds fewer than 2^32 threads)
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {       // (grid y: at most 65535 batch entries per launch)
        const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
        ColQuantArgs q = p;
        q.mat += b0 * n * m;
        if (q.row_scale && !q.bc) q.row_scale += b0 * n;
        q.scale += b0 * m;
        if (q.out_t) q.out_t += b0 * m * q.ld_t;
        if (q.out_n) q.out_n += b0 * n * q.ld_n;
        if (row_scale) {
            hipLaunchKernelGGL(k_col_scale_round_any, dim3((unsigned)col_tiles, (unsigned)nb), dim3(256), 0, (hipStream_t)stream, q);
            if (int e = launch_status()) return e;
            continue;
        }
        for (int64_t r0 = 0; r0 < row_tiles; r0 += per_launch) {
            const int64_t nr = row_tiles - r0 < per_launch ? row_tiles - r0 : per_launch;
            hipLaunchKernelGGL(k_col_round_any, dim3((unsigned)(col_tiles * nr), (unsigned)nb), dim3(256), 0, (hipStream_t)stream, q, (int32_t)col_tiles,
                               (int32_t)r0);
            if (int e = launch_status()) return e;
        }
    }
    return 0;
}

int cpmk_gemm_quantize_pair_ld(int64_t, const void*, void*, void*, int64_t, const void*, void*, void*, int32_t, int32_t, void*);   // quant.hip

int cpmk_gemm_quantize_cols_rows(int32_t batch, int32_t n, int32_t m, const void* mat, void* scale, void* out_t, int32_t ld_t, void* out_n, int32_t ld_n,
                                 int64_t rows, const void* row_mat, void* row_scale, void* row_out, void* stream) {
    clear_stale_error();
    if (rows < 0) return CPMK_EBADARG;
    if (n > 0 && batch > 0 && m > 0 && rows > 0 && scale && mat && out_t && ld_t >= n && ld_t % 16 == 0 && (!out_n || (ld_n >= m && (ld_n == m || ld_n % 16 == 0))) &&
        !any_null(row_mat, row_scale, row_out)) {
        const ColQuantArgs p = {n, m, (const half_t*)mat, nullptr, 0, (half_t*)scale, (int8_t*)out_t, (int8_t*)out_n, ld_t, out_n ? ld_n : 0};
        const RowQuantArgs r = {(const half_t*)row_mat, (half_t*)row_scale, (int8_t*)row_out, n, ld_t, rows, 0};
        const int rc = col_quantize<false>(batch, p, (hipStream_t)stream, &r);
        if (rc >= 0) return rc;
    }
    if (const int rc = cpmk_gemm_quantize_cols_ld(batch, n, m, mat, nullptr, 0, scale, out_t, ld_t, out_n, ld_n, stream)) return rc;
    return cpmk_gemm_quantize_pair_ld(rows, row_mat, row_scale, row_out, 0, nullptr, nullptr, nullptr, n, ld_t, stream);
}

int cpmk_gemm_backward_round_scale_ld(int32_t, int32_t, int32_t, const void*, const void*, void*, int32_t, void*, int, void*);       // train.hip

int cpmk_gemm_backward_quantize_both(int32_t batch, int32_t n, int32_t m, const void* mat, const void* row_scale, int broad_cast_row, void* scale, void* out_t, int32_t ld_t,
                                     const void* scale_y, int broad_cast_y, void* out, int32_t ld, void* scale_x, void* stream) {
    clear_stale_error();
    const int64_t rows = (int64_t)batch * n;
    if (n > 0 && batch > 0 && m > 0 && rows <= 0x7fffffff && ld_t >= n && ld_t % 16 == 0 && ld >= m && (ld == m || (ld % 16 == 0 && ld <= (m + 127) / 128 * 128)) &&
        !any_null(mat, row_scale, scale, out_t) && !any_null(scale_y, out, scale_x)) {
        const ColQuantArgs p = {n, m, (const half_t*)mat, (const half_t*)row_scale, broad_cast_row, (half_t*)scale, (int8_t*)out_t, nullptr, ld_t, 0};
        const RoundScaleArgs r = {(const half_t*)mat, (const half_t*)scale_y, (int8_t*)out, (half_t*)scale_x, rows, n, m, broad_cast_y, ld, 0};
        const int rc = col_quantize<true>(batch, p, (hipStream_t)stream, &r);
        if (rc >= 0) return rc;
    }
    if (const int rc = cpmk_gemm_backward_round_scale_ld(batch, n, m, mat, scale_y, out, ld, scale_x, broad_cast_y, stream)) return rc;
    if (row_scale == nullptr && rows > 0 && m > 0) return CPMK_EBADARG;       // (without rows there are no scales of theirs)
    return cpmk_gemm_quantize_cols_ld(batch, n, m, mat, row_scale, broad_cast_row, scale, out_t, ld_t, nullptr, 0, stream);
}

}  // extern "C"
