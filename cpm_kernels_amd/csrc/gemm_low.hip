// fp16 products of up to 64 output rows beside an operand stored (K, rows): attention's values x probabilities, and the gradients of queries
// and keys.  out[b, j, i] = sum_k P[b, j, k] Q[b, k, i], fp32 sums (cpm_kernels/torch/gemm.py:189-203).
//
// Bound by reading Q once.  A workgroup is one tile of 64 rows x 128 columns; it brings the next 64 rows of K into registers while
// the slab in LDS is multiplied, so pieces need no alignment, and four workgroups a compute unit have 96 KB in flight between them.
// Batch x depth x columns for 64 rows: 256 x 512 x 512 31.3 -> 30.8 us (5.4 TB/s), 512 of them 63.2 -> 58.7, 64 10.6 -> 8.8, 64 x 1024 x 1024 29 -> 27.3, 100 x 700 x 700 33.5 -> 28.1,
// 300 x 130 x 130 20.8 -> 7.4 (on the general kernel before), 128 x 400 x 400 13.5 -> 10.9.
#include "common.h"

namespace cpmk {

struct LowArgs {
    const half_t *P, *Q;           // (batch, n, k), (batch, k, m); a stride of 0 for one entry shared by the batch
    half_t* out;                   // (batch, n, m)
    int64_t strideP, strideQ;      // elements
    int32_t n, m, k;
    uint32_t tiles_c, tiles;
};

// NTH: Q in whole cache lines, read with the non-temporal hint.
template <bool NTH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_gemm_low(LowArgs a) {
    constexpr int TC = 128, SLAB = 64, RP = SLAB * 2, RQ = TC * 2;       // columns of the tile, depth of a slab, bytes per row in LDS
    __shared__ __attribute__((aligned(16))) int8_t lds[64 * RP + SLAB * RQ];
    int8_t* const ldsq = lds + 64 * RP;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4;
    const uint32_t t = xcd_remap(blockIdx.x, a.tiles);
    const uint32_t b = t / a.tiles_c, tc = t - b * a.tiles_c;
    // the last tile lies inside the matrix: what it shares with the one before is computed and stored twice, alike
    const int32_t i0 = min((int32_t)tc * TC, a.m - TC);
    const half_t* const Pb = a.P + b * a.strideP;
    const half_t* const Qb = a.Q + b * a.strideQ + i0;
    const int pr = tid >> 3, pc = tid & 7;                    // P: rows pr, pr + 32, piece pc of each (rows past n: the last one, not stored)
    const int lr = tid >> 4, lc = tid & 15;                   // Q: rows lr + 16 p of a slab, piece lc of each
    const uint32_t po0 = (uint32_t)min(pr, a.n - 1) * (uint32_t)a.k + pc * 8, po1 = (uint32_t)min(pr + 32, a.n - 1) * (uint32_t)a.k + pc * 8;
    auto load_q = [&](int32_t row) __attribute__((always_inline)) {
        const half_t* const src = Qb + ((uint32_t)row * (uint32_t)a.m + lc * 8);
        if constexpr (NTH) return __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(src));
        else return load_half8_any(src);
    };
    half8_t vp[2], vq[4];
    auto load = [&](int32_t k0) __attribute__((always_inline)) {
        if (k0 + SLAB <= a.k) {
            vp[0] = load_half8_any(Pb + (po0 + k0));
            vp[1] = load_half8_any(Pb + (po1 + k0));
#pragma unroll
            for (int p = 0; p < 4; ++p) vq[p] = load_q(k0 + lr + 16 * p);
        } else {            // the last a.k - k0 < SLAB of the depth, zeros behind them
            const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
            const int32_t left = a.k - k0 - pc * 8;           // of the piece and those behind it
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const half_t* const src = Pb + ((p ? po1 : po0) + k0);
                vp[p] = zero;
                if (left >= 8) vp[p] = load_half8_any(src);
                else if (left > 0) vp[p] = load_half8_head_any(src, left, zero);
            }
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                vq[p] = zero;
                if (k0 + lr + 16 * p < a.k) vq[p] = load_q(k0 + lr + 16 * p);
            }
        }
    };
    float4_t acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // P: piece c of row r at c ^ (r & 7), read 16 bytes at a time.  Q: transposing reads (ds_read_b64_tr_b16): within 16 lanes, lane j hands in the
    // address of four halves -- row of K k0 + j / 4, elements 4 (j % 4) .. + 3 of a block of 16 -- and lane i receives element i of rows
    // k0 .. k0 + 3; block u (32 bytes) of row k lies at u ^ (k & 3).
    const uint32_t qbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)ldsq + (q * 8 + (r16 >> 2)) * RQ + ((r16 & 3) << 3);
    auto frag_q = [&](int u, int ks) __attribute__((always_inline)) {
        typedef short short4_t __attribute__((ext_vector_type(4)));
        const uint32_t p0 = qbase + ks * 32 * RQ + (((u ^ (r16 >> 2)) & 3) << 5) + ((u >> 2) << 7);
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p0);
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)(p0 + 4 * RQ));
        return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    load(0);
    for (int32_t k0 = 0; k0 < a.k; k0 += SLAB) {
        if (k0 > 0) __syncthreads();                          // the slab before has been read
        *reinterpret_cast<half8_t*>(lds + pr * RP + ((pc ^ (pr & 7)) << 4)) = vp[0];
        *reinterpret_cast<half8_t*>(lds + (pr + 32) * RP + ((pc ^ (pr & 7)) << 4)) = vp[1];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int r = lr + 16 * p;
            *reinterpret_cast<half8_t*>(ldsq + r * RQ + (((lc >> 1) ^ (r & 3)) << 5) + ((lc & 1) << 4)) = vq[p];
        }
        __syncthreads();
        if (k0 + SLAB < a.k) load(k0 + SLAB);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            half8_t fp[4], fq[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) fp[i] = *reinterpret_cast<const half8_t*>(lds + (i * 16 + r16) * RP + (((ks * 4 + q) ^ (r16 & 7)) << 4));
#pragma unroll
            for (int j = 0; j < 2; ++j) fq[j] = frag_q(wave * 2 + j, ks);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[j], fp[i], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
    // Lane l, register e of a 16 x 16 result: output row l % 16, column (l / 16) * 4 + e.  The tile leaves through LDS in whole rows,
    // piece p of row r at p ^ (r & 15).
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[i][j][e];
            const int piece = wave * 4 + j * 2 + (q >> 1);
            *reinterpret_cast<half4_t*>(lds + (i * 16 + r16) * RQ + ((piece ^ r16) << 4) + ((q & 1) << 3)) = h;
        }
    __syncthreads();
    half_t* const ob = a.out + (int64_t)b * a.n * a.m + i0;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = lr + 16 * p;
        if (r < a.n) store_half8_any(ob + ((uint32_t)r * (uint32_t)a.m + lc * 8), *reinterpret_cast<const half8_t*>(lds + r * RQ + ((lc ^ (r & 15)) << 4)));
    }
}

// 0, an error code, or -1: not a product for this kernel.  A (batchA, k, m), B (batchB, n, k), out (batch, n, m).
int gemm_f16_low(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, const void* A, const void* B, void* out, hipStream_t st) {
    const int32_t batch = batchA > batchB ? batchA : batchB;
    // The tile kernel's workgroups of 256 columns and three slabs in flight are the better ones for deep products, which leave few workgroups (one of 64 x 1024 x
    // 1024 12.1 us, 11.1 here; 8 of 64 x 1500 x 1500 20.4 and 21.2; one of 64 x 8192 x 512 65 and 80), and where Q exceeds the last-level cache by far
    // (402 MB: 1024 of 64 x 1024 x 1024 443 and 457) or, in rows off cache lines, two thirds of it (168 MB: 1024 of 64 x 500 x 500 128.6 and 134; 300 of
    // them 43.3 and 42.8), unless its columns cover much more than the matrix (1024 of 64 x 300 x 300 67 and 58).
    if (n < 1 || n > 64 || m < 128 || k < 1 || k > 1024) return -1;
    const int64_t q = (int64_t)batchA * k * m, cover = ceil_div(m, 256) * 256;
    const bool lines = m % 64 == 0 && (reinterpret_cast<uintptr_t>(A) & 127u) == 0, wasteful = cover * 4 > ceil_div(m, 128) * 128 * 5;
    if (q > (lines ? 3ll << 26 : 5ll << 24) && !wasteful) return -1;
    // Off cache lines also beyond a depth of 512 where its tiles fill their rounds of the device (400 of 64 x 1000 x 200 47.3 and 54.2 us, 126 of 64 x 700 x
    // 900 37.5 and 40.5, 25 of 64 x 700 x 4454 37.3 and 40.0; 234 of 64 x 700 x 500, nearly two rounds, 39.5 and 42.5, 171 of them, a round and a third, 36.4 and 32.1), and
    // where it takes one of them for what are two tiles here, beyond a depth of 896 (150 of 64 x 1000 x 200 17.3 and 19, of 64 x 600 x 200 13.3 and 13.0).
    if (!lines && !wasteful && k > 512 && (m % 8 == 0 || m >= 256) && aligned16(A) && aligned16(B) && (reinterpret_cast<uintptr_t>(out) & 3u) == 0) {
        const int64_t cus = compute_units(), tiles = cover / 256 * batch, rounds = ceil_div(tiles, cus);
        if (rounds > 1 && tiles * 4 >= rounds * cus * 3) return -1;
        if (m < 256 && k > 896 && rounds == 1 && tiles * 5 >= cus * 2) return -1;
    }
    LowArgs a;
    a.P = (const half_t*)B; a.Q = (const half_t*)A; a.out = (half_t*)out;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k;
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k;
    a.n = n; a.m = m; a.k = k;
    const int64_t tc = ceil_div(m, 128);
    if (tc * batch >= 1 << 24 || (int64_t)n * k >= (1ll << 31) || (int64_t)m * (k + 64) >= (1ll << 31)) return -1;       // (a launch holds fewer than 2^32 threads)
    a.tiles_c = (uint32_t)tc; a.tiles = (uint32_t)(tc * batch);
    // (the hint where Q exceeds what the last-level cache keeps for its next reader: 512 of 64 x 512 x 512 58.1 us, 69 without; 256 of them
    // 28.4 and 29.8 by themselves, but the training step that reads Q again 528 and 524)
    if (lines && q >= 3ll << 25) hipLaunchKernelGGL(k_gemm_low<true>, dim3(a.tiles), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(k_gemm_low<false>, dim3(a.tiles), dim3(256), 0, st, a);
    return launch_status();
}

}  // namespace cpmk
