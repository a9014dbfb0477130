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
// The tile kernel also serves the fp16 products (gemm_f16.hip): the
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
    if (batchA == 1 && !bT && (srow == nullptr || !bcr) && (scol == nullptr || bcc) && rows_join(batch, n, k) &&
        rows_join_pays_i8(n, m, k, aT, batch, big_apart)) {
        n *= batch;
        batch = batchB = 1;
    }
    // (columns: operands that the tile kernel takes: it alone knows of `seg`)
    int32_t seg = 0;
    if (FUSED && batchB == 1 && aT && (srow == nullptr || bcr) && (scol == nullptr || !bcc) && cols_join(batch, m, k) && (int64_t)n * k < (1ll << 32) && aligned16(A) &&
        aligned16(B) && aligned16(out) && k > 0 && (bT ? k % 128 == 0 && n % 16 == 0 : k % 64 == 0) &&
        cols_join_pays_i8(n, m, k, !bT, batch, big_apart)) {
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
            // 128x128 tiles, or 128x64 when even those leave a quarter of the compute units idle, where these are one round, or two of them a compute unit and a
            // depth up to 768: 1208 x 2296, 180 tiles or 360, K = 128 7.3 us and 6.7, 512 8.5 and 8.0, 768 9.3 and 8.8, 4096 21.4 and 23.3 (operands out of memory
            // 8.0 and 7.2, 10.2 and 9.1, 11.3 and 10.7, 25.4 and 30.9); 500 x 5000, 160 or 316, K = 768 9.1 and 8.9 (11.5 and 11.6), 4096 20.6 and 27.4
            const int64_t mid = ceil_div(n, 128) * ceil_div(m, 128) * batch;
            // the smaller tiles finish a slab before a load from L2 returns: four ring stages keep them fed.  More
            // tiles than compute units but at most two each: a ring of two stages instead, which lets two
            // workgroups share a compute unit (2 x 80 KB of LDS) and all tiles run in one round, each
            // workgroup's waits covered by the other's MFMAs (6-11 % over 1.25-2 rounds of single workgroups)
            const int64_t cus = compute_units(), small = ceil_div(n, 128) * ceil_div(m, 64) * batch;
            if (mid * 4 >= cus * 3 || (small > cus && k > 768)) {
                if (mid > cus && mid <= 2 * cus) return launch_dma<2, 2, 2, 2, 128, EPI, 2, LAY, 32>(a, batch, st, 2);
                return launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, LAY, 32>(a, batch, st);
            }
            if (small > cus) return launch_dma<2, 2, 2, 1, 128, EPI, 2, LAY, 32>(a, batch, st, 2);
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
    if (seg) return CPMK_EBADARG;       // (never: joined products are the tile kernel's; below they would be written as one matrix)
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

}  // extern "C"
