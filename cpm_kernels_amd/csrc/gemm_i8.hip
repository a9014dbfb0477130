// int8 x int8 -> int32 batched GEMM on the CDNA4 matrix cores, optionally with the fp16
// dequantising epilogue applied to the accumulators in registers.
//
// Replaces the cuBLASLt call of the reference (cpm_kernels/kernels/gemm.py:127-186).  In
// row-major terms that call computes, per batch,
//     out[j, i] = sum_kk  Bop[j, kk] * Aop[i, kk]        j < n, i < m
// with Bop = B (n,k) if !bT else B^T of a (k,n) array, Aop = A^T of a (k,m) array if !aT
// else A (m,k).  Inside this file the operand indexed by the output ROW j is called P and
// the one indexed by the output COLUMN i is called Q; each is either "K-major" (kk
// contiguous) or "MN-major" (j resp. i contiguous).
//
// Three kernels, all exact (integer accumulation is order-independent, so the int32 result
// equals the reference's bit for bit):
//   k_gemm_dma     both operands K-major, k % 128 == 0: persistent workgroups walk the output
//                  tiles; global memory goes straight into a ring of XOR-swizzled LDS stages
//                  (global_load_lds_dwordx4), one barrier per 128-byte K slab, fragments read
//                  ahead of their MFMAs, v_mfma_i32_16x16x64_i8 (256x256 tiles) or
//                  v_mfma_i32_32x32x32_i8 (smaller tiles) with the operands swapped so that a lane
//                  owns 4 consecutive output columns; results leave through a per-wave LDS strip
//                  as whole 128-byte lines.
//                  With template parameter LAY it also takes operands stored with K as the row index
//                  (rows of whole 16-byte pieces), gathering the MFMA fragments element by element.
//   k_gemm_kmajor  both operands K-major, k % 16 == 0 (16-byte loads) or any k % 4 == 0 (4-byte loads): register-staged 64-byte K slabs.
//   k_gemm_generic any layout and size: LDS tiles + v_dot4_i32_i8.
// The tile kernel also serves the fp16 product of kernels/gemm.py:188-256 (cpmk_gemm_fp16): the
// same bytes of K per lane feed v_mfma_f32_16x16x32_f16 / v_mfma_f32_32x32x16_f16, with fp32 accumulators.
#include "gemm_tile.h"

namespace cpmk {

// ---------------------------------------------------------------------------------------
// Fast path
// ---------------------------------------------------------------------------------------
constexpr int BK = 64;   // bytes of K per LDS stage

// 16-byte chunk c (0..3) of LDS row r lives at chunk slot c ^ ((r >> 2) & 3): sixteen
// consecutive rows reading the same logical chunk then cover all 64 banks exactly once.
__device__ inline int lds_off(int r, int c) { return r * BK + ((c ^ ((r >> 2) & 3)) << 4); }

// DW: rows that are only 4-byte aligned (k % 16 != 0): a whole 16-byte piece still comes in one load (global loads of
// four dwords need dword alignment only), the piece across the end of K as single dwords, zero past the end.
struct __attribute__((aligned(4))) Int4Dword { int32_t x, y, z, w; };

template <int WAVES_R, int WAVES_C, int TR, int TC, bool FUSED, bool DW = false>
__global__ __launch_bounds__(WAVES_R* WAVES_C * 64) void k_gemm_kmajor(GemmArgs a) {
    constexpr int NT = WAVES_R * WAVES_C * 64;
    constexpr int BR = WAVES_R * TR * 32;   // output rows per workgroup
    constexpr int BC = WAVES_C * TC * 32;   // output columns per workgroup
    constexpr int CH_P = BR * (BK / 16) / NT;   // 16-byte chunks per thread, P tile
    constexpr int CH_Q = BC * (BK / 16) / NT;
    static_assert(BR * (BK / 16) % NT == 0 && BC * (BK / 16) % NT == 0, "tile/threads mismatch");

    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    constexpr int STAGE = (BR + BC) * BK;   // stage s: P tile at s*STAGE, Q tile after it

    // tile rasterisation: XCD-aware, then column-tile-fastest inside groups of 8 row tiles
    const uint32_t ntiles = (uint32_t)a.tiles_r * a.tiles_c;
    uint32_t t = xcd_remap(blockIdx.x, ntiles);
    constexpr uint32_t GR = 4;   // row tiles per raster group
    const uint32_t group_sz = GR * a.tiles_c;
    const uint32_t g = t / group_sz;
    const uint32_t rows_in_group = min(GR, (uint32_t)a.tiles_r - g * GR);
    const uint32_t tin = t - g * group_sz;
    const uint32_t tile_r = g * GR + tin % rows_in_group;
    const uint32_t tile_c = tin / rows_in_group;
    const int32_t j0 = tile_r * BR, i0 = tile_c * BC;

    const int b = blockIdx.z;
    const int8_t* P = a.P + (int64_t)b * a.strideP;
    const int8_t* Q = a.Q + (int64_t)b * a.strideQ;
    const int32_t K = a.k;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / WAVES_C, wc = wave % WAVES_C;

    // global -> register staging: chunk id q = tid + s*NT -> row q/4, chunk q%4
    int4_t gp[CH_P], gq[CH_Q];
    auto piece = [&](const int8_t* rowp, int32_t kc) __attribute__((always_inline)) {      // bytes [kc, kc + 16) of a row, zeros past K
        int4_t v = {0, 0, 0, 0};
        if constexpr (DW) {
            if (kc + 16 <= K) {
                const Int4Dword t = *reinterpret_cast<const Int4Dword*>(rowp + kc);
                v = int4_t{t.x, t.y, t.z, t.w};
            } else {
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (kc + 4 * d < K) v[d] = *reinterpret_cast<const int32_t*>(rowp + kc + 4 * d);
            }
        } else {
            if (kc < K) v = *reinterpret_cast<const int4_t*>(rowp + kc);
        }
        return v;
    };
    auto gload = [&](int32_t k0) {
#pragma unroll
        for (int s = 0; s < CH_P; ++s) {
            const int q = tid + s * NT, r = q >> 2, c = q & 3;
            const int32_t row = j0 + r;
            gp[s] = row < a.n ? piece(P + (int64_t)row * K, k0 + c * 16) : int4_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < CH_Q; ++s) {
            const int q = tid + s * NT, r = q >> 2, c = q & 3;
            const int32_t row = i0 + r;
            gq[s] = row < a.m ? piece(Q + (int64_t)row * K, k0 + c * 16) : int4_t{0, 0, 0, 0};
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int s = 0; s < CH_P; ++s) {
            const int q = tid + s * NT, r = q >> 2, c = q & 3;
            *reinterpret_cast<int4_t*>(smem + buf * STAGE + lds_off(r, c)) = gp[s];
        }
#pragma unroll
        for (int s = 0; s < CH_Q; ++s) {
            const int q = tid + s * NT, r = q >> 2, c = q & 3;
            *reinterpret_cast<int4_t*>(smem + buf * STAGE + BR * BK + lds_off(r, c)) = gq[s];
        }
    };

    int16_tv acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

    const int nk = (K + BK - 1) / BK;
    gload(0);
    sstore(0);
    __syncthreads();

    const int lrow = lane & 31, lk = lane >> 5;
    for (int it = 0; it < nk; ++it) {
        const int cur = it & 1;
        if (it + 1 < nk) gload((it + 1) * BK);
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            int4_t fa[TR], fb[TC];
#pragma unroll
            for (int i = 0; i < TR; ++i)
                fa[i] = *reinterpret_cast<const int4_t*>(smem + cur * STAGE + lds_off(wr * TR * 32 + i * 32 + lrow, ks * 2 + lk));
#pragma unroll
            for (int j = 0; j < TC; ++j)
                fb[j] = *reinterpret_cast<const int4_t*>(smem + cur * STAGE + BR * BK + lds_off(wc * TC * 32 + j * 32 + lrow, ks * 2 + lk));
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (it + 1 < nk) sstore(cur ^ 1);
        __syncthreads();
    }

    // epilogue: accumulator register e of lane l is output row (e/4)*8 + (l/32)*4 + e%4,
    // column l%32 of its 32x32 tile.
    const int64_t obase = (int64_t)b * a.n * a.m;
#pragma unroll
    for (int i = 0; i < TR; ++i) {
#pragma unroll
        for (int j = 0; j < TC; ++j) {
            const int32_t col = i0 + wc * TC * 32 + j * 32 + lrow;
            float sy = 0.0f;
            if (FUSED && col < a.m) sy = a.scol ? (float)a.scol[(a.bc_col ? 0 : (int64_t)b * a.m) + col] : 1.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int32_t row = j0 + wr * TR * 32 + i * 32 + (e >> 2) * 8 + lk * 4 + (e & 3);
                if (row < a.n && col < a.m) {
                    const int64_t o = obase + (int64_t)row * a.m + col;
                    if (FUSED) {
                        const float sx = a.srow ? (float)a.srow[a.bc_row ? row : (int64_t)b * a.n + row] : 1.0f;
                        reinterpret_cast<half_t*>(a.out)[o] = dequant(acc[i][j][e], sx, sy);
                    } else {
                        reinterpret_cast<int32_t*>(a.out)[o] = acc[i][j][e];
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------
// Generic path: 64x64 output tile, 32 bytes of K per stage, 256 threads each computing a
// 4x4 block with v_dot4_i32_i8.  Element-wise guarded loads handle every layout and size.
// ---------------------------------------------------------------------------------------
template <bool FUSED>
__global__ __launch_bounds__(256) void k_gemm_generic(GemmArgs a, int p_kmajor, int q_kmajor, int32_t row_base) {
    constexpr int T = 64, GK = 32, LD = GK + 4;
    __shared__ __attribute__((aligned(4))) int8_t sP[T * LD];
    __shared__ __attribute__((aligned(4))) int8_t sQ[T * LD];
    const int b = blockIdx.z;
    const int8_t* P = a.P + (int64_t)b * a.strideP;
    const int8_t* Q = a.Q + (int64_t)b * a.strideQ;
    const int32_t j0 = row_base + blockIdx.y * T, i0 = blockIdx.x * T;
    const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
    int32_t acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[r][c] = 0;

    for (int32_t k0 = 0; k0 < a.k; k0 += GK) {
#pragma unroll
        for (int s = 0; s < T * GK / 256; ++s) {
            const int q = tid + s * 256;
            int r, kk;
            if (p_kmajor) { r = q / GK; kk = q % GK; } else { r = q % T; kk = q / T; }
            const int32_t row = j0 + r, kg = k0 + kk;
            int8_t v = 0;
            if (row < a.n && kg < a.k) v = p_kmajor ? P[(int64_t)row * a.k + kg] : P[(int64_t)kg * a.n + row];
            sP[r * LD + kk] = v;
            if (q_kmajor) { r = q / GK; kk = q % GK; } else { r = q % T; kk = q / T; }
            const int32_t col = i0 + r, kg2 = k0 + kk;
            v = 0;
            if (col < a.m && kg2 < a.k) v = q_kmajor ? Q[(int64_t)col * a.k + kg2] : Q[(int64_t)kg2 * a.m + col];
            sQ[r * LD + kk] = v;
        }
        __syncthreads();
#pragma unroll
        for (int k4 = 0; k4 < GK / 4; ++k4) {
            int32_t pa[4], qb[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) pa[r] = *reinterpret_cast<const int32_t*>(sP + (ty * 4 + r) * LD + k4 * 4);
#pragma unroll
            for (int c = 0; c < 4; ++c) qb[c] = *reinterpret_cast<const int32_t*>(sQ + (tx + c * 16) * LD + k4 * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[r][c] = __builtin_amdgcn_sdot4(pa[r], qb[c], acc[r][c], false);
        }
        __syncthreads();
    }
    const int64_t obase = (int64_t)b * a.n * a.m;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int32_t row = j0 + ty * 4 + r;
        if (row >= a.n) continue;
        float sx = 0.0f;
        if (FUSED) sx = a.srow ? (float)a.srow[a.bc_row ? row : (int64_t)b * a.n + row] : 1.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int32_t col = i0 + tx + c * 16;
            if (col >= a.m) continue;
            const int64_t o = obase + (int64_t)row * a.m + col;
            if (FUSED) {
                const float sy = a.scol ? (float)a.scol[(a.bc_col ? 0 : (int64_t)b * a.m) + col] : 1.0f;
                reinterpret_cast<half_t*>(a.out)[o] = dequant(acc[r][c], sx, sy);
            } else {
                reinterpret_cast<int32_t*>(a.out)[o] = acc[r][c];
            }
        }
    }
}

template <int WAVES_R, int WAVES_C, int TR, int TC, bool FUSED, bool DW = false>
static int launch_kmajor(GemmArgs& a, int batch, hipStream_t st) {
    constexpr int BR = WAVES_R * TR * 32, BC = WAVES_C * TC * 32;
    constexpr int smem = 2 * (BR + BC) * BK;
    a.tiles_r = (int32_t)ceil_div(a.n, BR);
    a.tiles_c = (int32_t)ceil_div(a.m, BC);
    auto kern = k_gemm_kmajor<WAVES_R, WAVES_C, TR, TC, FUSED, DW>;
    static std::atomic<bool> lds_enabled[64];
    if (smem > 48 * 1024)
        if (int e = enable_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_enabled)) return e;
    dim3 grid((unsigned)(a.tiles_r * a.tiles_c), 1, (unsigned)batch);
    hipLaunchKernelGGL(kern, grid, dim3(WAVES_R * WAVES_C * 64), smem, st, a);
    return launch_status();
}

template <bool FUSED>
static int gemm_dispatch(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                         const void* A, const void* B, const void* srow, const void* scol, int bcr,
                         int bcc, void* out, hipStream_t st) {
    if (m < 0 || n < 0 || k < 0 || batchA < 1 || batchB < 1) return CPMK_EBADARG;
    if ((m % 4) || (n % 4) || (k % 4)) return CPMK_EALIGN;      // kernels/gemm.py:139
    if (!(batchA == batchB || batchA == 1 || batchB == 1)) return CPMK_EBADARG;   // :140
    int batch = batchA > batchB ? batchA : batchB;
    if (m == 0 || n == 0) return 0;
    if (out == nullptr || (k > 0 && any_null(A, B)) || (FUSED && srow == nullptr && scol == nullptr)) return CPMK_EBADARG;
    const int64_t big_apart = n > 128 && m > 128 ? ceil_div(n, 256) * ceil_div(m, 256) * batch : 0;       // (big_tiles)
    if (batchA == 1 && !bT && (srow == nullptr || !bcr) && (scol == nullptr || bcc) && rows_join(batch, n, k)) {
        n *= batch;
        batch = batchB = 1;
    }
    // (columns: where whole entries of them leave tiles half empty)
    int32_t seg = 0;
    if (FUSED && batchB == 1 && aT && (srow == nullptr || bcr) && (scol == nullptr || !bcc) && cols_join(batch, m, k) && aligned16(A) && aligned16(B) && aligned16(out) &&
        k > 0 && (bT ? k % 128 == 0 && n % 16 == 0 : k % 64 == 0) &&
        (ceil_div((int64_t)m * batch, 128) < ceil_div(m, 128) * batch || ceil_div((int64_t)m * batch, 256) < ceil_div(m, 256) * batch)) {
        seg = m;
        m *= batch;
        batch = batchA = 1;
    }
    if (batch > 65535) {      // some kernels index the batch with the grid's z dimension: at most 65535 entries per call
        constexpr int64_t ESZ_OUT = FUSED ? 2 : 4;
        for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
            const int32_t nb = (int32_t)(batch - b0 < 65535 ? batch - b0 : 65535);
            const int rc = gemm_dispatch<FUSED>(
                m, k, n, batchA == 1 ? 1 : nb, batchB == 1 ? 1 : nb, aT, bT,
                (const int8_t*)A + (batchA == 1 ? 0 : b0 * m * k), (const int8_t*)B + (batchB == 1 ? 0 : b0 * n * k),
                srow ? (const half_t*)srow + (bcr ? 0 : b0 * n) : nullptr, scol ? (const half_t*)scol + (bcc ? 0 : b0 * m) : nullptr,
                bcr, bcc, (int8_t*)out + b0 * n * m * ESZ_OUT, st);
            if (rc != 0) return rc;
        }
        return 0;
    }
    GemmArgs a;
    a.P = (const int8_t*)B; a.Q = (const int8_t*)A; a.out = out;
    a.srow = (const half_t*)srow; a.scol = (const half_t*)scol;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k;
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k;
    a.n = n; a.m = m; a.k = k; a.bc_row = bcr; a.bc_col = bcc;
    a.tiles_r = a.tiles_c = 0;
    a.edge_in = 0;
    a.nsum = 1;
    a.kmagic = 0;
    a.seg = seg;
    a.segmagic = seg ? (uint32_t)(((1ull << 32) + seg - 1) / seg) : 0;
    // the tile kernel stores 16-byte pieces of output rows (8-byte halves where fp16 rows are not whole pieces: m % 8 == 4)
    const bool wide = aligned16(out);
    const bool p_kmajor = !bT, q_kmajor = aT != 0;
    const bool fast = p_kmajor && q_kmajor && k > 0 && (k % 16 == 0) && aligned16(A) && aligned16(B);
    if (fast && wide && (k % 64 == 0) && (int64_t)n * k < (1ll << 32) && (int64_t)m * k < (1ll << 32)) {
        // 256x256 tiles when they give most compute units a tile, else 128x128
        const int64_t big = big_tiles(n, m, batch, big_apart);
        constexpr int EPI = FUSED ? kEpiDequant : kEpiInt32;
        auto kmajor = [&](auto lay) __attribute__((always_inline)) {
            constexpr int LAY = decltype(lay)::value;
            if (k % 128 != 0) {
                // a depth of whole 64-byte but not whole 128-byte slabs (1600, 4544 ...): the same kernels on 64-byte slabs and
                // a ring of four stages -- twice the barriers per byte of K, 5-10 % behind the 128-byte form
                if (big * 4 >= compute_units() * 3 && n > 128 && m > 128) return launch_dma<2, 4, 4, 2, 64, EPI, 4, LAY, 16>(a, batch, st);
                return launch_dma<2, 2, 2, 2, 64, EPI, kRingSmall, LAY, 32>(a, batch, st);
            }
            // (a dimension of at most 128 would leave half or more of every 256-wide tile empty)
            if (big * 4 >= compute_units() * 3 && n > 128 && m > 128) return launch_dma<2, 4, 4, 2, 128, EPI, kRingBig, LAY, 16>(a, batch, st);
            // 128x128 tiles, or 128x64 when even those leave a quarter of the compute units idle and twice as many of half their size are one round
            // (two workgroups a compute unit of the latter: 500 x 5000, 160 tiles or 320, K = 4096 23.5 us, 18.5 so; K = 12160 58 and 43; K = 512 8.1 and 8.0)
            const int64_t mid = ceil_div(n, 128) * ceil_div(m, 128) * batch;
            // the smaller tiles finish a slab before a load from L2 returns: four ring stages keep them fed.  More
            // tiles than compute units but at most two each: a ring of two stages instead, which lets two
            // workgroups share a compute unit (2 x 80 KB of LDS) and all tiles run in one round, each
            // workgroup's waits covered by the other's MFMAs (6-11 % over 1.25-2 rounds of single workgroups)
            const int64_t cus = compute_units(), small = ceil_div(n, 128) * ceil_div(m, 64) * batch;
            if (mid * 4 >= cus * 3 || small > cus) {
                if (mid > cus && mid <= 2 * cus) return launch_dma<2, 2, 2, 2, 128, EPI, 2, LAY, 32>(a, batch, st, 2);
                return launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, LAY, 32>(a, batch, st);
            }
            return launch_dma<2, 2, 2, 1, 128, EPI, kRingSmall, LAY, 32>(a, batch, st);
        };
        if constexpr (FUSED) {
            if (seg) return kmajor(std::integral_constant<int, 16>{});
        }
        return kmajor(std::integral_constant<int, 0>{});
    }
    // a depth that is not whole 64-byte slabs (4000, 4048, 4100 ...): the tile kernels on 64-byte slabs, the rest of the
    // depth straight from memory into the fragments (k % 4 == 0 is the reference's precondition: rows of whole dwords)
    if (p_kmajor && q_kmajor && wide && k > 64 && (k % 4 == 0) && (reinterpret_cast<uintptr_t>(A) & 3u) == 0 &&
        (reinterpret_cast<uintptr_t>(B) & 3u) == 0 && (int64_t)n * k < (1ll << 32) && (int64_t)m * k < (1ll << 32)) {
        constexpr int EPI = FUSED ? kEpiDequant : kEpiInt32;
        const int64_t big = big_tiles(n, m, batch, big_apart);
        const bool large = big * 4 >= compute_units() * 3 && n > 128 && m > 128;
        if (fast) return large ? launch_dma<2, 4, 4, 2, 64, EPI, 4, 4, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 64, EPI, kRingSmall, 4, 32>(a, batch, st);
        return large ? launch_dma<2, 4, 4, 2, 64, EPI, 4, 12, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 64, EPI, kRingSmall, 12, 32>(a, batch, st);
    }
    // an operand stored (K, rows): the tile kernel reads it as it lies and takes the fragments with transposing LDS reads
    // (rows of such an operand that are not whole 16-byte pieces: tiles that stay inside the matrix, which takes a matrix of
    // at least one tile)
    const bool in_p = !p_kmajor && n % 16 != 0, in_q = !q_kmajor && m % 16 != 0;
    if (!(p_kmajor && q_kmajor) && wide && k > 0 && (k % 128 == 0) && aligned16(A) && aligned16(B) && (!in_p || n >= 128) &&
        (!in_q || m >= 128) && (int64_t)n * k < (1ll << 32) && (int64_t)m * k < (1ll << 32)) {
        constexpr int EPI = FUSED ? kEpiDequant : kEpiInt32;
        // 256x256 tiles when they give most compute units a tile, else 128x128 (as for K-major operands)
        const int64_t big = big_tiles(n, m, batch, big_apart);
        const bool large = big * 4 >= compute_units() * 3 && n > 128 && m > 128 && (!in_p || n >= 256) && (!in_q || m >= 256);
        a.edge_in = (in_p ? 1 : 0) | (in_q ? 2 : 0);
        if constexpr (FUSED) {
            if (seg) return large ? launch_dma<2, 4, 4, 2, 128, EPI, 2, 17, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 17, 32>(a, batch, st);
        }
        switch ((p_kmajor ? 0 : 1) | (q_kmajor ? 0 : 2)) {
            case 1: return large ? launch_dma<2, 4, 4, 2, 128, EPI, 2, 1, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 1, 32>(a, batch, st);
            case 2: return large ? launch_dma<2, 4, 4, 2, 128, EPI, 2, 2, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 2, 32>(a, batch, st);
            default: return large ? launch_dma<2, 4, 4, 2, 128, EPI, 2, 3, 16>(a, batch, st) : launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 3, 32>(a, batch, st);
        }
    }
    // one operand stored (K, rows) and a depth beyond one slab that is not whole slabs: the 32x32 form of the tile kernel,
    // the rest of the depth as a slab filled up with zeros
    if (p_kmajor != q_kmajor && wide && k > 128 && (k % 4 == 0) && aligned16(A) && aligned16(B) && (!in_p || n >= 128) &&
        (!in_q || m >= 128) && (int64_t)n * k < (1ll << 32) && (int64_t)m * k < (1ll << 32)) {
        constexpr int EPI = FUSED ? kEpiDequant : kEpiInt32;
        a.edge_in = (in_p ? 1 : 0) | (in_q ? 2 : 0);
        if (!p_kmajor) return launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 13, 32>(a, batch, st);
        return launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, 14, 32>(a, batch, st);
    }
    if (fast) {
        const int64_t t256 = ceil_div(n, 256) * ceil_div(m, 128) * batch;
        if (t256 >= 256) return launch_kmajor<2, 2, 4, 2, FUSED>(a, batch, st);
        return launch_kmajor<2, 2, 2, 2, FUSED>(a, batch, st);
    }
    // K-major rows that are only 4-byte aligned (k % 16 != 0; k % 4 == 0 always): the same kernel on 4-byte loads
    if (p_kmajor && q_kmajor && k > 0 && batch <= 65535 && (reinterpret_cast<uintptr_t>(A) & 3u) == 0 && (reinterpret_cast<uintptr_t>(B) & 3u) == 0 &&
        (FUSED ? (reinterpret_cast<uintptr_t>(out) & 1u) == 0 : (reinterpret_cast<uintptr_t>(out) & 3u) == 0)) {
        const int64_t t256 = ceil_div(n, 256) * ceil_div(m, 128) * batch;
        if (t256 >= 256) return launch_kmajor<2, 2, 4, 2, FUSED, true>(a, batch, st);
        return launch_kmajor<2, 2, 2, 2, FUSED, true>(a, batch, st);
    }
    // output rows are the grid's y dimension (65535 tiles of 64 rows): taller products go out in several launches
    for (int64_t r0 = 0; r0 < n; r0 += 65535ll * 64) {
        const int64_t nr = n - r0 < 65535ll * 64 ? n - r0 : 65535ll * 64;
        dim3 grid((unsigned)ceil_div(m, 64), (unsigned)ceil_div(nr, 64), (unsigned)batch);
        hipLaunchKernelGGL((k_gemm_generic<FUSED>), grid, dim3(256), 0, st, a, (int)p_kmajor, (int)q_kmajor, (int32_t)r0);
        if (int e = launch_status()) return e;
    }
    return 0;
}

// ---------------------------------------------------------------------------------------
// fp16 product (fp32 accumulation), any layout, size and alignment: 64x64 output tile, 64 halves of K per
// stage, four waves of one 32x32 MFMA tile each.  Shapes that are whole slabs and pieces run on the tile
// kernel above instead.
// ---------------------------------------------------------------------------------------
// V: halves per global access (4, 2 or 1: what the contiguous dimension of both operands and the alignment of the buffers allow).
template <int V>
__global__ __launch_bounds__(256) void k_gemm_f16_generic(GemmArgs a, int p_kmajor, int q_kmajor, int32_t row_base) {
    // Guarded loads bring a 64 x 64 piece of each operand into LDS with K contiguous (zeros past the edges,
    // so any size, layout and alignment works); each of the four waves then owns a 32 x 32 quarter of the tile and
    // multiplies with v_mfma_f32_32x32x16_f16.
    constexpr int T = 64, GK = 64, LD = GK + 4;        // rows of 136 bytes: 8-byte aligned fragment reads, spread over the banks
    __shared__ __attribute__((aligned(16))) half_t sP[T * LD];
    __shared__ __attribute__((aligned(16))) half_t sQ[T * LD];
    const int b = blockIdx.z;
    const int32_t k = a.k >> 1;                        // a.k is the row length in bytes
    const half_t* P = reinterpret_cast<const half_t*>(a.P + (int64_t)b * a.strideP);
    const half_t* Q = reinterpret_cast<const half_t*>(a.Q + (int64_t)b * a.strideQ);
    const int32_t j0 = row_base + blockIdx.y * T, i0 = blockIdx.x * T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int lrow = lane & 31, lk = lane >> 5;
    float16_tv acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    typedef _Float16 halfV_t __attribute__((ext_vector_type(V > 1 ? V : 2)));
    // V halves of one operand's piece: along K for a K-major operand (one row), along the rows for one stored (K, rows).
    // A stage's pieces are requested one stage ahead into registers, so that their latency passes under the products.
    constexpr int S = T * GK / V / 256;       // accesses per thread, operand and stage
    auto place = [&](int kmajor, int q, int& r, int& kk) __attribute__((always_inline)) {
        if (kmajor) { r = q / (GK / V); kk = (q % (GK / V)) * V; } else { r = (q % (T / V)) * V; kk = q / (T / V); }
    };
    auto fetch = [&](half_t (&v)[V], const half_t* G, int kmajor, int32_t r0, int32_t L, int32_t k0, int q) __attribute__((always_inline)) {
        int r, kk;
        place(kmajor, q, r, kk);
        const int32_t row = r0 + r, kg = k0 + kk;
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = (half_t)0.0f;
        if (row < L && kg < k) {            // (L and k are multiples of V where the access runs along them)
            const half_t* src = kmajor ? G + ((int64_t)row * k + kg) : G + ((int64_t)kg * L + row);
            if constexpr (V > 1) {
                const halfV_t t = *reinterpret_cast<const halfV_t*>(src);
#pragma unroll
                for (int e = 0; e < V; ++e) v[e] = t[e];
            } else {
                v[0] = *src;
            }
        }
    };
    auto put = [&](half_t* sm, const half_t (&v)[V], int kmajor, int q) __attribute__((always_inline)) {
        int r, kk;
        place(kmajor, q, r, kk);
#pragma unroll
        for (int e = 0; e < V; ++e) sm[kmajor ? r * LD + kk + e : (r + e) * LD + kk] = v[e];
    };
    half_t rp[S][V], rq[S][V];
    auto fetch_all = [&](int32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            fetch(rp[s], P, p_kmajor, j0, a.n, k0, tid + s * 256);
            fetch(rq[s], Q, q_kmajor, i0, a.m, k0, tid + s * 256);
        }
    };
    fetch_all(0);
    for (int32_t k0 = 0; k0 < k; k0 += GK) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            put(sP, rp[s], p_kmajor, tid + s * 256);
            put(sQ, rq[s], q_kmajor, tid + s * 256);
        }
        __syncthreads();
        if (k0 + GK < k) fetch_all(k0 + GK);
#pragma unroll
        for (int ks = 0; ks < GK / 16; ++ks) {
            // lane (lrow, lk): the 8 halves k = 16 ks + 8 lk .. + 7 of its row / column, as two 8-byte reads
            const half_t* pp = sP + (wr * 32 + lrow) * LD + ks * 16 + lk * 8;
            const half_t* qp = sQ + (wc * 32 + lrow) * LD + ks * 16 + lk * 8;
            const half4_t p0 = *reinterpret_cast<const half4_t*>(pp), p1 = *reinterpret_cast<const half4_t*>(pp + 4);
            const half4_t q0 = *reinterpret_cast<const half4_t*>(qp), q1 = *reinterpret_cast<const half4_t*>(qp + 4);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_shufflevector(p0, p1, 0, 1, 2, 3, 4, 5, 6, 7),
                                                         __builtin_shufflevector(q0, q1, 0, 1, 2, 3, 4, 5, 6, 7), acc, 0, 0, 0);
        }
        __syncthreads();
    }
    // accumulator register e of lane l: output row (e / 4) * 8 + (l / 32) * 4 + e % 4, column l % 32 of the wave's quarter
    const int64_t obase = (int64_t)b * a.n * a.m;
    const int32_t col = i0 + wc * 32 + lrow;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int32_t row = j0 + wr * 32 + (e >> 2) * 8 + lk * 4 + (e & 3);
        if (row < a.n && col < a.m) reinterpret_cast<half_t*>(a.out)[obase + (int64_t)row * a.m + col] = (half_t)acc[e];
    }
}

static int gemm_f16_dispatch(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                             const void* A, const void* B, void* out, hipStream_t st) {
    if (m < 0 || n < 0 || k < 0 || batchA < 1 || batchB < 1) return CPMK_EBADARG;
    if ((m % 2) || (n % 2) || (k % 2)) return CPMK_EALIGN;      // kernels/gemm.py:200
    if (!(batchA == batchB || batchA == 1 || batchB == 1)) return CPMK_EBADARG;   // :201
    int batch = batchA > batchB ? batchA : batchB;
    if (m == 0 || n == 0) return 0;
    if (out == nullptr || (k > 0 && any_null(A, B))) return CPMK_EBADARG;
    if (k > (1 << 30)) return CPMK_ETOOBIG;
    const int64_t big_apart = n > 128 && m > 128 ? ceil_div(n, 256) * ceil_div(m, 256) * batch : 0;       // (big_tiles)
    if (batchA == 1 && !bT && rows_join(batch, n, (int64_t)k * 2)) {
        n *= batch;
        batch = batchB = 1;
    }
    if (batch > 65535) {      // (grid z: at most 65535 batch entries per call)
        for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
            const int32_t nb = (int32_t)(batch - b0 < 65535 ? batch - b0 : 65535);
            const int rc = gemm_f16_dispatch(m, k, n, batchA == 1 ? 1 : nb, batchB == 1 ? 1 : nb, aT, bT,
                                             (const half_t*)A + (batchA == 1 ? 0 : b0 * m * k), (const half_t*)B + (batchB == 1 ? 0 : b0 * n * k),
                                             (half_t*)out + b0 * n * m, st);
            if (rc != 0) return rc;
        }
        return 0;
    }
    GemmArgs a;
    a.P = (const int8_t*)B; a.Q = (const int8_t*)A; a.out = out;
    a.srow = nullptr; a.scol = nullptr;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k * 2;          // bytes
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k * 2;
    a.n = n; a.m = m; a.k = k * 2; a.bc_row = 0; a.bc_col = 0;
    a.tiles_r = a.tiles_c = 0;
    a.edge_in = 0;
    a.nsum = 1;
    a.kmagic = 0;
    a.seg = 0;
    a.segmagic = 0;
    // The tile kernel stores 16-byte pieces of output rows that start on dwords, and 8-byte halves at a row's end.  Rows of 4j + 2
    // elements end in neither: their last column tile lies inside the matrix (edge_in), which takes a matrix of at least one tile.
    const bool odd = m % 4 != 0;
    // (The line at 192 columns was drawn for depths up to 128 with both operands stored (K, rows), which have a kernel of their own now; what it still keeps on
    // the general kernel is deeper or stored otherwise and would mostly be quicker on the tiles from 128 columns on: 80 of 150 x 150, both stored (K, rows),
    // K = 256 22.6 us and 8.6, K = 512 42.6 and 12.2; both K-major, K = 512 15.8 and 11.4, 300 of 130 x 130, K = 1000 84 and 103.)
    const bool wide = (reinterpret_cast<uintptr_t>(out) & 3u) == 0 && (!odd || m >= 192);
    const bool p_kmajor = !bT, q_kmajor = aT != 0;
    // A depth up to 128: a kernel of its own -- but where the output's rows are not whole cache lines and it exceeds half of the last-level
    // cache, the tile kernel, whose large tiles share fewer of the lines (1024 of 500 x 500, K = 64 149 us, 162 there; 100 of 1000 x 1000 52.6 and
    // 56.4; 250 of 500 x 500 32.7 and 25.1), unless those cover much more than the matrix (1500 of 300 x 300 179 and 113).  And the tile kernel
    // too, beyond a quarter of that cache, where its large tiles cover no more than the small ones do, of which the last overlap the ones before
    // them: for depths of two slabs (7659 of 136 x 192, K = 128 217 us, 245 there; 976 of 200 x 1024 145 and 161; 5425 of 192 x 192 187 and 199), and
    // for an operand shared by the batch that is one large tile, of one whole slab or of two (2034 of 192 x 512 with the 192 shared, K = 64 104 and
    // 119; with the 512 shared 111 and 68; 976 of 400 x 512, the 400 shared, 106 and 71), or of two if it is the row operand (the same, K = 128, 134 and 146).
    if (!p_kmajor && !q_kmajor && k > 0 && k <= 128) {
        const int64_t big = ceil_div(n, 256) * ceil_div(m, 256), mid = ceil_div(n, 128) * ceil_div(m, 128), area = (int64_t)n * m, outs = batch * area;
        const bool large = big * 8 <= mid * 3 && big * batch * 4 >= (int64_t)compute_units() * 3;
        const bool exact = big * 4 == mid && (n % 8 == 0 || n >= 256) && (m % 8 == 0 || m >= 256) && wide && aligned16(A) && aligned16(B);
        const bool overlap = batchA == batchB ? k > 112 && mid * 65536 > 5 * area
                                              : mid * 131072 > 9 * area && (batchB == 1 ? k > 112 || (k == 64 && n <= 256) : m <= 256 && (k == 64 || k > 112));
        if (!large || ((m % 64 == 0 || outs <= 1 << 26) && !(exact && overlap && outs > 1 << 25)))
            if (const int rc = gemm_f16_short(m, k, n, batchA, batchB, A, B, out, st); rc >= 0) return rc;
    }
    if (p_kmajor && !q_kmajor && n <= 64 && k > 0)       // probabilities x values
        if (const int rc = gemm_f16_low(m, k, n, batchA, batchB, A, B, out, st); rc >= 0) return rc;
    if (p_kmajor && q_kmajor && wide && k > 0 && (k % 32 == 0) && aligned16(A) && aligned16(B) &&
        (int64_t)n * k * 2 < (1ll << 32) && (int64_t)m * k * 2 < (1ll << 32)) {
        const int64_t big = big_tiles(n, m, batch, big_apart);
        const bool whole128 = k % 64 == 0;       // the depth is whole 128-byte slabs (else whole 64-byte ones: 96, 160 ...)
        a.edge_in = odd ? 2 : 0;
        if (big * 4 >= compute_units() * 3 && n > 128 && m > 128 && (!odd || m >= 256)) {
            if (whole128 && k >= 256) return launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 0, 16>(a, batch, st);
            // Products of a few slabs -- attention scores, K = 64 -- are all prologue and epilogue, bound by the stores (and
            // depths of whole 64-byte slabs only need this form anyway):
            // the 32x32 form is quicker there, and waves of 64 rows x 128 columns, whose row segments are 256 bytes,
            // store 5-15 % faster than waves of 128 x 64 (slabs of 64 bytes make room for their wider output strips)
            return launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, 0, 32>(a, batch, st);
        }
        if (!whole128) return launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, 0, 32>(a, batch, st);
        // (as for int8: more 128x128 tiles than compute units but at most two each -> two workgroups per compute unit)
        const int64_t mid = ceil_div(n, 128) * ceil_div(m, 128) * batch, cus = compute_units();
        if (mid > cus && mid <= 2 * cus) return launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 0, 32>(a, batch, st, 2);
        return launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 0, 32>(a, batch, st);
    }
    // a depth that is not whole 64-byte slabs (K = 40, 72, 500, 1000 ...): the same kernels, the rest of the depth straight
    // from memory into the fragments (large tiles) or as a slab filled up with zeros
    if (p_kmajor && q_kmajor && wide && k > 32 && (reinterpret_cast<uintptr_t>(A) & 3u) == 0 && (reinterpret_cast<uintptr_t>(B) & 3u) == 0 &&
        (int64_t)n * k * 2 < (1ll << 32) && (int64_t)m * k * 2 < (1ll << 32)) {
        const int64_t big = big_tiles(n, m, batch, big_apart);
        const bool large = big * 4 >= compute_units() * 3 && n > 128 && m > 128 && (!odd || m >= 256);
        a.edge_in = odd ? 2 : 0;
        if (k % 8 == 0 && aligned16(A) && aligned16(B))       // whole, aligned 16-byte pieces
            return large ? launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, 4, 32>(a, batch, st) : launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, 4, 32>(a, batch, st);
        return large ? launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, 12, 32>(a, batch, st) : launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, 12, 32>(a, batch, st);
    }
    // an operand stored (K, rows): the tile kernel reads it as it lies, with transposing LDS reads for the fragments
    // (rows of such an operand that are not whole 16-byte pieces: tiles that stay inside the matrix, which takes a matrix of at
    // least one tile)
    const bool in_p = !p_kmajor && n % 8 != 0, in_q = !q_kmajor && m % 8 != 0;
    // 64 x 256 tiles for few output rows (attention: probabilities x values)
    const bool low = n <= 64 && !((in_q || odd) && m < 256);
    if (!(p_kmajor && q_kmajor) && wide && k >= 64 && aligned16(A) && aligned16(B) &&
        (!in_p || n >= 128) && (!in_q || m >= (low ? 256 : 128)) &&
        (int64_t)n * k * 2 < (1ll << 32) && (int64_t)m * k * 2 < (1ll << 32)) {
        const int lay = (p_kmajor ? 0 : 1) | (q_kmajor ? 0 : 2);
        // 256x256 tiles when they give most compute units a tile, else 128x128 (as for K-major operands) -- and when the
        // larger ones cover over half as much again as the smaller ones do, where that costs more than their better ratio of products to reads
        // saves: 300 x 300 over 400 heads, both stored (K, rows), K = 512 140 us with large tiles, 120 us with small ones, K = 160 70 and 46 us;
        // 580 x 580 (1.44 times the area) alike; with one operand K-major and K = 80 70 us with large tiles, 74 us with small ones.
        const int64_t big = ceil_div(n, 256) * ceil_div(m, 256), mid = ceil_div(n, 128) * ceil_div(m, 128);
        // (not where the large tiles are one round of the device: 384 x 384 over 50 heads, K = 1024 28 us with large tiles, 38 us with small ones)
        const int64_t cus = compute_units();
        const bool waste = big * 8 > mid * 3 && (lay == 3 || k >= 256) && big * batch > cus;
        // At depths that are not whole slabs no last round is split into half tiles, and whole rounds of the device count: a large tile takes
        // as long as two to two and a half small ones (3592 x 384 over 4 entries, K = 8576 and the rest 8: two rounds of large tiles 226 us,
        // four of small ones 181; 1792 x 384 x 24, K = 3592: 257 and 219).
        const bool rest = k % 64 != 0;       // (see below)
        const bool idle = rest && k >= 256 && ceil_div(big * batch, cus) * 9 > ceil_div(mid * batch, cus) * 4;
        const bool large = !waste && !idle && big_tiles(n, m, batch, big_apart) * 4 >= cus * 3 && n > 128 && m > 128 && (!in_p || n >= 256) &&
                           (!(in_q || odd) || m >= 256);
        a.edge_in = (in_p ? 1 : 0) | (in_q || odd ? 2 : 0);
        // a depth that is not whole slabs (probabilities x values over 500 keys, scores over heads of 80): its rest is a slab
        // filled up with zeros
        // more 128x128 tiles than compute units but at most two each: two workgroups a compute unit, as for K-major operands (2460 x 384 over
        // 7 entries, K = 6144, 420 tiles: 144 -> 120 us; 300 tiles of 640 x 640, K = 2048: 50 -> 37 us)
        const bool two = mid * batch > cus && mid * batch <= 2 * cus;
        switch (lay) {
            case 1:
                if (low) return rest ? launch_dma<1, 4, 2, 2, 128, kEpiF16, 3, 13, 32>(a, batch, st) : launch_dma<1, 4, 2, 2, 128, kEpiF16, 3, 1, 32>(a, batch, st);
                if (large) return rest ? launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 13, 16>(a, batch, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 1, 16>(a, batch, st);
                return rest ? launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 13, 32>(a, batch, st)
                     : two ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 1, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 1, 32>(a, batch, st);
            case 2:
                if (low) return rest ? launch_dma<1, 4, 2, 2, 128, kEpiF16, 3, 14, 32>(a, batch, st) : launch_dma<1, 4, 2, 2, 128, kEpiF16, 3, 2, 32>(a, batch, st);
                if (large) return rest ? launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 14, 16>(a, batch, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 2, 16>(a, batch, st);
                return rest ? launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 14, 32>(a, batch, st)
                     : two ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 2, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 2, 32>(a, batch, st);
            default:
                if (low && !rest) return launch_dma<1, 4, 2, 2, 128, kEpiF16, 3, 3, 32>(a, batch, st);
                if (large) return rest ? launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 15, 16>(a, batch, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 3, 16>(a, batch, st);
                return rest ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 15, 32>(a, batch, st, 2)
                     : two ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 3, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 3, 32>(a, batch, st);
        }
    }
    for (int64_t r0 = 0; r0 < n; r0 += 65535ll * 64) {        // (rows beyond the grid's y dimension: several launches)
        const int64_t nr = n - r0 < 65535ll * 64 ? n - r0 : 65535ll * 64;
        dim3 grid((unsigned)ceil_div(m, 64), (unsigned)ceil_div(nr, 64), (unsigned)batch);
        // the widest access both operands allow: their contiguous dimension a multiple of it, their buffers aligned to it
        const int32_t cp = p_kmajor ? k : n, cq = q_kmajor ? k : m;
        const uintptr_t al = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B);
        if (cp % 4 == 0 && cq % 4 == 0 && (al & 7u) == 0)
            hipLaunchKernelGGL(k_gemm_f16_generic<4>, grid, dim3(256), 0, st, a, (int)p_kmajor, (int)q_kmajor, (int32_t)r0);
        else if (cp % 2 == 0 && cq % 2 == 0 && (al & 3u) == 0)
            hipLaunchKernelGGL(k_gemm_f16_generic<2>, grid, dim3(256), 0, st, a, (int)p_kmajor, (int)q_kmajor, (int32_t)r0);
        else
            hipLaunchKernelGGL(k_gemm_f16_generic<1>, grid, dim3(256), 0, st, a, (int)p_kmajor, (int)q_kmajor, (int32_t)r0);
        if (int e = launch_status()) return e;
    }
    return 0;
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_gemm_int8(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                   const void* A, const void* B, void* out, void* stream) {
    clear_stale_error();
    return gemm_dispatch<false>(m, k, n, batchA, batchB, aT, bT, A, B, nullptr, nullptr, 0, 0, out,
                                (hipStream_t)stream);
}

int cpmk_gemm_int8_scale(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                         const void* A, const void* B, const void* scale_row, const void* scale_col,
                         int broad_cast_row, int broad_cast_col, void* out, void* stream) {
    clear_stale_error();
    if ((int64_t)n * m > 0 && any_null(scale_row, scale_col)) return CPMK_EBADARG;
    return gemm_dispatch<true>(m, k, n, batchA, batchB, aT, bT, A, B, scale_row, scale_col, broad_cast_row,
                               broad_cast_col, out, (hipStream_t)stream);
}

int cpmk_gemm_int8_scale_one(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                             const void* A, const void* B, const void* scale_row, const void* scale_col,
                             int broad_cast_row, int broad_cast_col, void* out, void* stream) {
    clear_stale_error();
    return gemm_dispatch<true>(m, k, n, batchA, batchB, aT, bT, A, B, scale_row, scale_col, broad_cast_row,
                               broad_cast_col, out, (hipStream_t)stream);
}

int cpmk_gemm_fp16(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                   const void* A, const void* B, void* out, void* stream) {
    clear_stale_error();
    return gemm_f16_dispatch(m, k, n, batchA, batchB, aT, bT, A, B, out, (hipStream_t)stream);
}

}  // extern "C"
