// fp16 products of a depth up to 128, both operands stored (K, rows): attention scores k^T q, and the gradient of the probabilities,
// from (batch * heads, head, seq) tensors.  out[b, j, i] = sum_k P[b, k, j] Q[b, k, i], fp32 sums
// (cpm_kernels/torch/gemm.py:189-203).
//
// Bound by writing the output.  The persistent tile kernel (gemm_tile.h) alternates between its stores and everything else, one
// 256 x 256 tile a compute unit at a time, in row segments of 128 bytes; here a workgroup is one 128 x 128 tile that takes 32 KB of LDS -- a slab of
// the operands first, the output later -- and 128 registers a lane, so that four of them on a compute unit load, multiply and store at
// different times, and the segments are 256 bytes.  Heads of seq x seq, K = 64: 256 of 512 32.1 -> 26.6 us (6.3 TB/s), 64 of 512 13.0 -> 9.7,
// 1024 of 300 111 -> 66, 250 of 500 32.7 -> 25.1, 1024 of 1024 513 -> 485; K = 80, 256 of 512 41 -> 33; K = 40 50 -> 25.
#include "common.h"

namespace cpmk {

struct ShortArgs {
    const half_t *P, *Q;           // (batch, k, n), (batch, k, m); a stride of 0 for one entry shared by the batch
    half_t* out;                   // (batch, n, m)
    int64_t strideP, strideQ;      // elements
    int32_t n, m, k;
    uint32_t tiles_r, tiles_c, tiles;
};

// NTS: the output is stored with the non-temporal hint.
// WHOLE: the tiles do not overlap.  Elsewhere the last ones leave out the rows, and the whole pieces of them, that the tiles before store (6510 of
// 160 x 192, K = 64 203 us with them written again, 145 so; with the choice also where nothing overlaps 1024 of 1024 x 1024 527 us, 513 so).
template <bool NTS, bool WHOLE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_gemm_short(ShortArgs a) {
    constexpr int T = 128, SLAB = 64, ROW = T * 2;            // tile edge, rows of K at a time, bytes per row in LDS
    __shared__ __attribute__((aligned(16))) int8_t lds[2 * SLAB * ROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4, wr = wave >> 1, wc = wave & 1;
    // column tiles of a row of tiles follow one another on one XCD: they share cache lines where rows of the output are not whole ones
    const uint32_t t = xcd_remap(blockIdx.x, a.tiles);
    const uint32_t b = t / (a.tiles_r * a.tiles_c), rest = t - b * (a.tiles_r * a.tiles_c), tr = rest / a.tiles_c, tc = rest - tr * a.tiles_c;
    // the last tiles lie inside the matrix: what they share with the tiles before them is computed twice, alike, but stored once
    const int32_t j0 = min((int32_t)tr * T, a.n - T), i0 = min((int32_t)tc * T, a.m - T);
    const half_t* const Pb = a.P + b * a.strideP + j0;
    const half_t* const Qb = a.Q + b * a.strideQ + i0;
    const int lr = tid >> 4, lc = tid & 15;                   // rows lr + 16 p of a slab, 16-byte piece lc of each
    half8_t v[8];
    auto load = [&](int32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            v[p] = load_half8_any(Pb + ((uint32_t)(k0 + lr + 16 * p) * (uint32_t)a.n + lc * 8));
            v[4 + p] = load_half8_any(Qb + ((uint32_t)(k0 + lr + 16 * p) * (uint32_t)a.m + lc * 8));
        }
    };
    auto load_rest = [&](int32_t k0) __attribute__((always_inline)) {       // the last a.k - k0 < SLAB rows, zeros behind them
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            v[p] = v[4 + p] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
            if (k0 + lr + 16 * p < a.k) {
                v[p] = load_half8_any(Pb + ((uint32_t)(k0 + lr + 16 * p) * (uint32_t)a.n + lc * 8));
                v[4 + p] = load_half8_any(Qb + ((uint32_t)(k0 + lr + 16 * p) * (uint32_t)a.m + lc * 8));
            }
        }
    };
    float4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // Transposing reads (ds_read_b64_tr_b16): within 16 lanes, lane j hands in the address of four halves -- row of K k0 + j / 4, elements
    // 4 (j % 4) .. + 3 of a block of 16 -- and lane i receives element i of rows k0 .. k0 + 3.  Block u (32 bytes) of row k lies at u ^ (k & 3),
    // which spreads a wave's reads over the banks.
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)lds;
    const uint32_t frag0 = base + (q * 8 + (r16 >> 2)) * ROW + ((r16 & 3) << 3);
    auto frag = [&](int operand, int u, int ks) __attribute__((always_inline)) {
        typedef short short4_t __attribute__((ext_vector_type(4)));
        const uint32_t p0 = frag0 + operand * SLAB * ROW + ks * 32 * ROW + (((u ^ (r16 >> 2)) & 3) << 5) + ((u >> 2) << 7);
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p0);
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)(p0 + 4 * ROW));
        return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    for (int32_t k0 = 0; k0 < a.k; k0 += SLAB) {
        if (k0 + SLAB <= a.k) load(k0);                       // (requested while the slab before is multiplied it costs registers that a fourth workgroup needs)
        else load_rest(k0);
        if (k0 > 0) __syncthreads();                          // the slab before has been read
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int r = lr + 16 * p;
            int8_t* const dst = lds + r * ROW + (((lc >> 1) ^ (r & 3)) << 5) + ((lc & 1) << 4);
            *reinterpret_cast<half8_t*>(dst) = v[p];
            *reinterpret_cast<half8_t*>(dst + SLAB * ROW) = v[4 + p];
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            half8_t fp[4], fq[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) fp[i] = frag(0, wr * 4 + i, ks);
#pragma unroll
            for (int j = 0; j < 4; ++j) fq[j] = frag(1, wc * 4 + j, ks);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[j], fp[i], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
    // Lane l, register e of a 16 x 16 result: output row l % 16, column (l / 16) * 4 + e.  The tile is put together in LDS,
    // piece p of row r at p ^ (r & 15), and leaves in whole rows.
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[i][j][e];
            const int piece = wc * 8 + j * 2 + (q >> 1);
            *reinterpret_cast<half4_t*>(lds + (wr * 64 + i * 16 + r16) * ROW + ((piece ^ r16) << 4) + ((q & 1) << 3)) = h;
        }
    __syncthreads();
    half_t* const ob = a.out + ((int64_t)b * a.n + j0) * a.m + i0;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int r = lr + 16 * p;
        if constexpr (!WHOLE)
            if (r < (int32_t)tr * T - j0 || lc * 8 + 8 <= (int32_t)tc * T - i0) continue;
        const half8_t h = *reinterpret_cast<const half8_t*>(lds + r * ROW + ((lc ^ (r & 15)) << 4));
        half_t* const dst = ob + (int64_t)r * a.m + lc * 8;
        if constexpr (NTS) __builtin_nontemporal_store(h, reinterpret_cast<half8_t*>(dst));
        else store_half8_any(dst, h);
    }
}

// 0, an error code, or -1: not a product for this kernel.  A (batchA, k, m), B (batchB, k, n), out (batch, n, m).
int gemm_f16_short(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, const void* A, const void* B, void* out, hipStream_t st) {
    const int32_t batch = batchA > batchB ? batchA : batchB;
    if (n < 128 || m < 128 || k < 1 || k > 128) return -1;
    ShortArgs a;
    a.P = (const half_t*)B; a.Q = (const half_t*)A; a.out = (half_t*)out;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k;
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k;
    a.n = n; a.m = m; a.k = k;
    const int64_t tr = ceil_div(n, 128), tc = ceil_div(m, 128);
    if (tr * tc * batch >= 1 << 24 || (int64_t)n * k >= (1ll << 31) || (int64_t)m * k >= (1ll << 31)) return -1;       // (a launch holds fewer than 2^32 threads)
    a.tiles_r = (uint32_t)tr; a.tiles_c = (uint32_t)tc; a.tiles = (uint32_t)(tr * tc * batch);
    // Whole cache lines and more of them than the last-level cache holds beside what is read: 512 of 512 x 512 52 us with the hint, 70 without,
    // 400 of them 41 and 47, 1024 of 1024 x 1024 485 and 516; 256 of 512 x 512, which the next kernel finds in the cache, 26.6 either way.
    const bool lines = m % 64 == 0 && (reinterpret_cast<uintptr_t>(out) & 127u) == 0, large = (int64_t)batch * n * m >= 3ll << 25;
    const bool whole = n % 128 == 0 && m % 128 == 0;
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(a.tiles), dim3(256), 0, st, a); };
    if (lines && large) go(whole ? k_gemm_short<true, true> : k_gemm_short<true, false>);
    else go(whole ? k_gemm_short<false, true> : k_gemm_short<false, false>);
    return launch_status();
}

}  // namespace cpmk
