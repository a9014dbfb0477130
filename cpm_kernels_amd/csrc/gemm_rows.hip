// fp16 products of a depth up to 80 in rows off cache lines, both operands stored (K, rows): attention scores k^T q, and the gradient of the
// probabilities, of sequences that are no multiple of 64.  out[b, j, i] = sum_k P[b, k, j] Q[b, k, i], fp32 sums
// (cpm_kernels/torch/gemm.py:189-203).
//
// Bound by writing the output.  Tiles of part of a row write segments that begin and end inside cache lines, which their neighbours complete at
// another time.  Here a workgroup has whole rows, a multiple of 16 and as many as LDS holds at most (about 1200 at K <= 32, 400 at K = 80): 16 at a time are put together in LDS as they lie in memory and leave as whole aligned
// lines.  A wave has 128 columns, whose operand it keeps in registers, transposed there, for all rows of the workgroup.
// Heads of seq x seq, K = 64, with operands that are not in the caches and a pass over the output behind (of 186 us for 1024 of 500, 63 for 300, which is in both figures):
// 1024 of 500 330 -> 290 us, 512 158 -> 133, 128 45 -> 40, 1024 of 300 131 -> 115, 100 of 902 114 -> 86; 1024 of 110 38 -> 28, 32 14.8 -> 9.7; K = 80 66 of 902 81 -> 72,
// 900 of 70 33 -> 21.  Stores with the non-temporal hint are quicker by themselves (1024 of 500 161 -> 94 us over operands in the cache), but leave the next
// kernel nothing there (334 us with the pass behind for 64 rows a workgroup, 320 with the hint; 256 rows 292 and 298; 512 of 500 139 and 156).
#include "common.h"
#include <type_traits>

namespace cpmk {

struct RowsArgs {
    const half_t *P, *Q;           // (batch, k, n), (batch, k, m); a stride of 0 for one entry shared by the batch
    half_t* out;                   // (batch, n, m), 16-byte aligned; n, m even
    int64_t strideP, strideQ;      // elements
    int32_t n, m, k;
    int32_t tall;                  // rows of a workgroup, a multiple of 16
    uint32_t chunks, items;        // workgroups of an entry, of all
};

// Eight rows of K from k0 on (zeros beyond K), elements c .. c + 7 of each, as eight pieces along K.  Every load is made, at a row inside the operand,
// so that none waits for another.
__device__ __forceinline__ void load_block8(half8_t (&v)[8], const half_t* base, int32_t L, int32_t k, int32_t k0, int32_t c) {
    const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = load_half8_any(base + (int64_t)min(k0 + u, k - 1) * L + c);
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (k0 + u >= k) v[u] = zero;
    transpose_half8x8(v);
}

// KS: k-steps of 32.  AL: bytes on which every eighth element of the output's rows starts (16, 8 or 4).
template <int KS, int AL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(KS == 3 ? 3 : 4, KS == 3 ? 3 : 4))) void k_gemm_rows(RowsArgs a) {
    extern __shared__ __attribute__((aligned(16))) int8_t rows_lds[];
    const int32_t tall = a.tall;
    int8_t* const pl = rows_lds;                                   // P: 16 bytes for eight of K of a row; row r of K-piece kb at kb * tall + (r ^ (r / 8) % 8)
    int8_t* const strip = rows_lds + tall * KS * 64;
    const int tid = threadIdx.x, lane = tid & 63, NT = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const uint32_t t = xcd_remap(blockIdx.x, a.items);
    const uint32_t b = t / a.chunks;
    const int32_t j0 = (int32_t)(t - b * a.chunks) * tall, rows = min(tall, a.n - j0);
    const half_t* const Pb = a.P + b * a.strideP;
    const half_t* const Qb = a.Q + b * a.strideQ;
    for (int i = tid; i < tall / 8 * KS * 4; i += NT) {
        const int rb = i % (tall / 8), kb = i / (tall / 8);
        // (the last blocks of rows and of columns lie inside the matrix and repeat some of those before them)
        const int32_t at = min(j0 + rb * 8, a.n - 8) - j0;
        if (at + 8 <= rb * 8) continue;
        half8_t v[8];
        load_block8(v, Pb, a.n, a.k, kb * 8, j0 + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int r = at + e;
            if (r >= 0) *reinterpret_cast<half8_t*>(pl + (kb * tall + (r ^ ((r >> 3) & 7))) * 16) = v[e];
        }
    }
    // fragment e of the wave: element e of 16 blocks of eight columns
    const int32_t c0 = wave * 128;
    half8_t fq[KS][8];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) load_block8(fq[ks], Qb, a.m, a.k, ks * 32 + q * 8, min(c0 + r16 * 8, a.m - 8));
    const int64_t first = ((int64_t)b * a.n + j0) * a.m * 2;       // bytes
    const int32_t pitch = a.m * 2;
    uint4_t kept = {0, 0, 0, 0};
    __syncthreads();
    for (int32_t r0 = 0; r0 < rows; r0 += 16) {
        float4_t acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int r = r0 + r16;
            const half8_t fp = *reinterpret_cast<const half8_t*>(pl + ((ks * 4 + q) * tall + (r ^ ((r >> 3) & 7))) * 16);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[ks][e], fp, acc[e], 0, 0, 0);
        }
        int8_t* const dst = reinterpret_cast<int8_t*>(a.out) + first + (int64_t)r0 * pitch;
        const int32_t lead = (int32_t)(reinterpret_cast<uintptr_t>(dst) & 127u), end = lead + min(16, rows - r0) * pitch;       // in the strip, multiples of 8
        if (r0 > 0) {
            __syncthreads();                                       // the rows before have been read
            if (tid < 8) {                                         // the line that they began
                if (tid * 16 < lead) *reinterpret_cast<uint2_t*>(strip + tid * 16) = uint2_t{kept[0], kept[1]};
                if (tid * 16 + 8 < lead) *reinterpret_cast<uint2_t*>(strip + tid * 16 + 8) = uint2_t{kept[2], kept[3]};
            }
        }
        // Lane l, register g of fragment e: row l % 16, element e of block (l / 16) * 4 + g
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int32_t c = c0 + (q * 4 + g) * 8;
            half8_t h;
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = (half_t)acc[e][g];
            int8_t* const at = strip + lead + r16 * pitch + min(c, a.m - 8) * 2;
            const uint4_t w = __builtin_bit_cast(uint4_t, h);
            if (c < a.m) {
                if constexpr (AL == 16) {
                    *reinterpret_cast<uint4_t*>(at) = w;
                } else if constexpr (AL == 8) {
                    *reinterpret_cast<uint2_t*>(at) = uint2_t{w[0], w[1]};
                    *reinterpret_cast<uint2_t*>(at + 8) = uint2_t{w[2], w[3]};
                } else {
#pragma unroll
                    for (int d = 0; d < 4; ++d) *reinterpret_cast<uint32_t*>(at + d * 4) = w[d];
                }
            }
        }
        __syncthreads();
        const bool last = r0 + 16 >= rows;
        const int32_t from = r0 == 0 ? lead : 0, upto = last ? end : end & ~127;
        int8_t* const line = dst - lead;
        for (int32_t o = tid * 16; o < upto; o += NT * 16) {
            const uint4_t w = *reinterpret_cast<const uint4_t*>(strip + o);
            if (o >= from && o + 16 <= upto) {
                *reinterpret_cast<uint4_t*>(line + o) = w;
            } else {
                if (o >= from) *reinterpret_cast<uint2_t*>(line + o) = uint2_t{w[0], w[1]};
                if (o + 8 >= from && o + 16 <= upto) *reinterpret_cast<uint2_t*>(line + o + 8) = uint2_t{w[2], w[3]};
            }
        }
        if (tid < 8) kept = *reinterpret_cast<const uint4_t*>(strip + min((end & ~127) + tid * 16, end & ~15));
    }
}

// Rows of a workgroup, a multiple of 16, at most the 80 KB of LDS that two workgroups a compute unit leave each: the fewest rounds of the device, of eight waves a compute unit at least (twelve of short rows), times the time of one, its start as long as 200
// rows (1024 of 500 x 500 in one, two and four parts 289, 293 and 309 us, 128 of them 58, 45 and 40, 256 81, 72 and 73; 186 of 572 x 572
// in two, three and four 71, 79 and 74, 150 of 570 x 570 62, 58 and 64).
static int32_t rows_tall(int32_t n, int32_t m, int ks, int64_t batch) {
    const int64_t cus = compute_units(), waves = ceil_div(m, 128), floor = waves >= 4 ? 2 : 12 / waves, cap = (80 * 1024 - 128 - 32ll * m) / (ks * 64) / 16 * 16;
    const int64_t least = ceil_div(n, cap);
    int64_t best = 0, best_t = 0;
    for (int64_t parts = least; parts == least || (parts <= ceil_div(n, 32) && parts < least + 32); ++parts) {
        const int64_t tall = ceil_div(ceil_div(n, parts), 16) * 16, each = ceil_div(ceil_div(n, tall) * batch, cus), t = (each > floor ? each : floor) * (tall + 200);
        if (best == 0 || t < best_t) {
            best = tall;
            best_t = t;
        }
    }
    return (int32_t)best;
}

// 0, an error code, or -1: not a product for this kernel.  A (batchA, k, m), B (batchB, k, n), out (batch, n, m).
int gemm_f16_rows(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, const void* A, const void* B, void* out, hipStream_t st) {
    const int64_t batch = batchA > batchB ? batchA : batchB;
    if (m <= 64 || m > 1024 || m % 64 == 0 || n < 8 || k < 1 || k > 80 || m % 2 || n % 2 || !aligned16(out)) return -1;
    // Outputs of 38 MB and more, with three k-steps 50 unless the rows are short, from where the workgroups' start is hidden (the other kernels and this one, timed as above:
    // 128 of 500 x 500 45 / 40 us, 64 of them 24.4 / 26.6; 200 of 300 x 300 33 / 30, 64 of them 15 / 17; 48 of 700 x 700 36 / 34; 800 of 150 x 150 38 / 34, 64 of them
    // 9.6 / 11.3; K = 80 50 of 600 x 600 32 / 35, 528 of 154 x 154 34 / 30), and any number where the matrix is smaller than the other kernels' tiles (100 of 100 x 100 13.6 / 11.1,
    // 32 of 110 x 110 14.8 / 9.7, 400 of 120 x 120 17.6 / 17.1).  Whole lines stay where they are (512 of 256 x 256 45 / 52, 128 of 512 x 512 43 / 46), and tall matrices of
    // less than a wave's columns (512 of 500 x 80 42 / 47).
    const bool large = m > 128 && batch * n * m >= (k <= 64 ? 9ll << 21 : m <= 256 ? 3ll << 22 : 3ll << 23), little = n > 64 && n < 128 && m < 128;
    if (!large && !little) return -1;
    RowsArgs a;
    a.P = (const half_t*)B; a.Q = (const half_t*)A; a.out = (half_t*)out;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k;
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k;
    a.n = n; a.m = m; a.k = k;
    const int ks = (int)ceil_div(k, 32);
    a.tall = rows_tall(n, m, ks, batch);
    const int64_t chunks = ceil_div(n, a.tall), nt = ceil_div(m, 128) * 64;
    if (chunks * batch * nt >= 1ll << 32) return -1;       // (a launch holds fewer than 2^32 threads)
    a.chunks = (uint32_t)chunks; a.items = (uint32_t)(chunks * batch);
    const int lds = a.tall * ks * 64 + 128 + 16 * m * 2;
    int rc = 0;
    auto go = [&](auto ksc, auto alc) {
        auto kern = k_gemm_rows<decltype(ksc)::value, decltype(alc)::value>;
        static std::atomic<bool> lds_enabled[64];
        rc = enable_dynamic_lds(reinterpret_cast<const void*>(kern), 80 * 1024, lds_enabled);
        if (rc == 0) hipLaunchKernelGGL(kern, dim3(a.items), dim3((unsigned)nt), (unsigned)lds, st, a);
    };
    auto steps = [&](auto alc) {
        if (ks == 1) go(std::integral_constant<int, 1>{}, alc);
        else if (ks == 2) go(std::integral_constant<int, 2>{}, alc);
        else go(std::integral_constant<int, 3>{}, alc);
    };
    if (m % 8 == 0) steps(std::integral_constant<int, 16>{});
    else if (m % 4 == 0) steps(std::integral_constant<int, 8>{});
    else steps(std::integral_constant<int, 4>{});
    return rc != 0 ? rc : launch_status();
}

}  // namespace cpmk
