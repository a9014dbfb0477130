// Products summed over the batch:  out[g, j, i] = sum over the entries e of group g of  P[e, j, :] . Q[e, i, :]
// -- the gradient of an operand that the forward product broadcast over the batch (a weight), which the reference forms
// as one product per entry followed by a sum over them (cpm_kernels/torch/gemm.py:115-186, 219-239).
#include "gemm_tile.h"

namespace cpmk {

// ---------------------------------------------------------------------------------------
// Products summed over the batch
// ---------------------------------------------------------------------------------------
// Partial sums a product of (n, m) outputs over `batch` entries is formed in: as few as give most compute units a tile,
// a divisor of the batch, and at most kSumMax entries each (the int8 form keeps their scales in a 4 KB strip).
constexpr int kSumMax = 16;
static int32_t sum_groups(int32_t m, int32_t n, int32_t batch) {
    const int64_t cus = compute_units(), tiles = ceil_div(n, 128) * ceil_div(m, 128);
    for (int32_t g = 1; g < batch; ++g)
        if (batch % g == 0 && batch / g <= kSumMax && tiles * g * 4 >= cus * 3) return g;
    return batch;
}

// Groups for products of depth k an entry, or `batch` where the products one by one and their sum are the quicker: a product in large
// tiles makes up for writing and adding its output where the sum over the batch has too few outputs for such tiles and
// multiplies in small ones.  The sums / entries in us on either side of each line (outputs x batch x k):
//   int8       one group   8192 x 1024 x 7: k = 2048 111 / 132, 4096 247 / 242; 4096 x 4096 x 8: 3072 359 / 422, 4096 578 / 517
//              several     1536 x 1536 x 12: 896 49 / 50, 1536 67 / 62
//   fp16, large tiles      4096 x 4096 x 2: k = 34 ... 4096 all quicker; 4096 x 4096 x 8: 4096 806 / 902
//   fp16 K-major, one      2560 x 2560 x 5: 384 50 / 50, 448 54 / 48;  k of whole 16-byte pieces 328 52 / 53, 392 62 / 58;  others 66 38 / 42, 140 51 / 45
//              several     1536 x 1536 x 12: 256 38 / 41, 384 53 / 44;  pieces 72 30 / 38, 136 41 / 40;  others 66 57 / 42
//   fp16 (K, rows), one    2560 x 2560 x 5: 576 55 / 56, 768 73 / 67
//              several     1536 x 1536 x 12: 256 36 / 41, 384 47 / 46
enum SumKind { kSumI8 = 0, kSumF16 = 1, kSumF16KFirst = 2 };
static int32_t sum_groups_for(int kind, int32_t m, int32_t k, int32_t n, int32_t batch) {
    int32_t g = sum_groups(m, n, batch);
    // (K, rows): a group's entries become one contraction, which the tile kernel takes up to operands of 4 GiB
    if (kind == kSumF16KFirst)
        while (g < batch && (int64_t)(m > n ? m : n) * k >= (1ll << 31) / (batch / g))
            do ++g; while (batch % g != 0);
    if (g == batch) return batch;
    const int64_t cus = compute_units();
    const bool one = g == 1, large = ceil_div(n, 256) * ceil_div(m, 256) * g * 4 >= cus * 3;
    if (kind != kSumI8) {
        // A last round of few tiles idles most of the device for a whole batch's depth, where the single products have one at the
        // end of all entries: at least three quarters of the rounds are to be filled (a last round of up to half the device is half tiles,
        // where the depth is whole slabs).  5376 x 896 x 16, k = 68, 294 small
        // tiles: 121 us summed, 77 one by one; 3328 x 5376 x 12, k = 2048, 273 large ones: the training step 2403 and 2145 us.
        const int64_t tiles = (large ? ceil_div(n, 256) * ceil_div(m, 256) : ceil_div(n, 128) * ceil_div(m, 128)) * g, r = tiles % cus;
        const int64_t halves = tiles / cus * 2 + (r == 0 ? 0 : 2 * r <= cus && tiles > cus && k % 64 == 0 ? 1 : 2);
        if (tiles * 8 < cus * 3 * halves) return batch;
    }
    int32_t limit;
    if (kind == kSumI8) limit = one ? 2048 : 1024;
    else if (large) return g;
    else if (kind == kSumF16KFirst) limit = one ? 576 : 256;
    else if (k % 32 == 0) limit = one ? 384 : 256;
    else if (k % 8 == 0) limit = one ? 328 : 96;
    else limit = one ? 96 : 0;
    return k <= limit ? g : batch;
}

// Products of up to 512 tiles of 128 x 128 (fp16: of too few large ones): the number of groups of the least of these estimates, in us, whether it fills the device or
// not.  Fitted to 900 sizes of 4 to 4096 a side, 2 to 64 entries and depths of 32 to 2048; the choice over the best number for each as a geometric mean, int8
// 1.017, fp16 K-major 1.012 (23 of 271 and 15 of 317 more than a tenth slower than the best; the lines above, which ask for a tile a compute unit, 1.05 and 1.06).
// Groups / one by one: int8 512 x 512 x 2, k = 128 7 / 16; x 13, 128 15 / 22; 832 x 1856 x 7, 128 11 / 23; x 16, 512 30 (two groups) / 39; 384 x 64 x 5, 256 11.7 / 9.5 (the
// second launch costs the host more);
// fp16 1280 x 3328 x 14, k = 48 28 / 54; 512 x 512 x 6, 512 36 / 14 (one by one).
// One by one: entries of at least half a round of the device's two tiles a compute unit, and no less than results written and read at 5.2 TB/s and products at
// 4.4 (2.0) PFLOP/s take.
static float sum_apart_time(bool i8, int64_t cus, int64_t tiles, int32_t m, int32_t k, int32_t n, int32_t batch) {
    const float rounds = (float)(tiles * batch) / (float)(2 * cus), slabs = (float)ceil_div((int64_t)k * (i8 ? 1 : 2), 128), out = (float)batch * (float)n * (float)m * 1e-6f;
    const float part = rounds > 1.0f ? (i8 ? 0.69f : 0.91f) * rounds : (i8 ? 0.67f : 0.73f) * (rounds > 0.5f ? rounds : 0.5f);
    const float t = (i8 ? 9.1f : 9.4f) + slabs * part + (i8 ? 0.16f : 0.35f) * out + (i8 ? 7.8f : 5.4f) * rounds;
    const float least = (i8 ? 12.0f : 9.0f) + out * (4.0f / 5.2f + 2.0f * (float)k / (i8 ? 4400.0f : 2000.0f));
    return t > least && out * (float)k <= 75000.0f ? t : least;        // (the first is not fitted to more than 1.5e11 operations, where large tiles are quicker than it says)
}
// A group: 4.5, and for each of its entries 0.40 and 0.45 a slab of 128 bytes (int8: folding, products), or 0.65 a slab (fp16; depths that are not whole
// ones 0.7 and 0.26 a 64-byte slab, 2.0 and 0.30 where rows are not whole 16-byte pieces), half as much again where int8 tiles share compute units, a round of the
// device after the other for fp16; several groups 3 and their fp32 sums at 4.7 TB/s.
static float sum_group_time(bool i8, int64_t cus, int64_t tiles, int32_t m, int32_t k, int32_t n, int32_t batch, int32_t g) {
    const int64_t work = tiles * g, last = work % cus;
    const float area = (float)n * (float)m * 1e-6f, kb = (float)(i8 ? k : 2 * k);
    const bool slabs = i8 || k % 64 == 0;
    const float entry = i8 ? 0.40f + 0.45f * ceilf(kb / 128.0f) : slabs ? 0.65f * kb / 128.0f : k % 8 == 0 ? 0.7f + 0.26f * floorf(kb / 64.0f) : 2.0f + 0.30f * floorf(kb / 64.0f);
    float rounds;
    if (i8) rounds = work <= cus ? 1.0f : 1.5f * (float)ceil_div(work, 2 * cus);
    else rounds = (float)(work / cus) + (last == 0 ? 0.0f : 2 * last <= cus && work > cus && slabs ? 0.5f : 1.0f);
    return 4.5f + rounds * (float)(batch / g) * entry + (g > 1 ? 3.0f + (float)g * area * 8.0f / 4.7f : 0.0f);
}

// (K, rows): whether the tile kernel takes the groups (gemm_rows_parts), else the kernel for any size does
static bool krows_tiles(int32_t m, int64_t depth, int32_t n) { return depth >= 64 && (n % 8 == 0 || n >= 128) && (m % 8 == 0 || m >= 256); }
// The entries of a group are one contraction of operands below 4 GiB; one group's is a product like any other (krows_time), whose depth may be divided.
static float sum_krows_time(int64_t cus, int64_t tiles, int32_t m, int32_t k, int32_t n, int32_t batch, int32_t g) {
    const int64_t depth = (int64_t)k * (batch / g);
    if ((m > n ? m : n) * depth >= 1ll << 31) return 1e30f;
    if (g == 1) return krows_time(m, (int32_t)depth, n);
    const float slabs = (float)ceil_div(depth, 64), add = 3.0f + (float)g * (float)n * (float)m * 8e-6f / 4.7f;
    if (krows_tiles(m, depth, n)) {
        const float rounds = (float)(tiles * g) / (float)cus;
        return 4.5f + add + slabs * (depth % 64 == 0 ? 0.47f : 0.55f) * (rounds <= 1.0f ? 1.0f : rounds <= 2.0f ? 2.05f : 1.15f * rounds);
    }
    const float rounds = (float)(ceil_div(n, 64) * ceil_div(m, 64) * g) / (float)cus;
    return 2.6f + add + slabs * (rounds <= 1.0f ? 0.58f : rounds <= 4.0f ? 1.1f : 0.29f * rounds);
}
static bool sum_few_tiles(int kind, int64_t cus, int32_t m, int32_t n) {
    return ceil_div(n, 128) * ceil_div(m, 128) <= 2 * cus && (kind == kSumI8 || ceil_div(n, 256) * ceil_div(m, 256) * 4 < cus * 3);
}

// (K, rows): groups, the batch's entries one by one among them, whose sums stay fp32; 0: one by one, rounded, from the depths on where that is the quicker.  One contraction
// of all entries whatever its depth had left a few tiles with one slab after another: 8 x 44 outputs, 26 entries of k = 128 30.8 us, 28 x 8 x 24, 980 200 us; as the 26 and the 24
// groups of one entry 6.5 and 13.8 (one by one 9.9 and 17.1); 136 x 890 x 49, 128 50 us, seven groups 17.0 (20.7); 1644 x 2132 x 10, 512 in one 54 (75)
static int32_t sum_krows_groups(int32_t m, int32_t k, int32_t n, int32_t batch) {
    const int64_t cus = compute_units(), tiles = ceil_div(n, 128) * ceil_div(m, 128);
    if (!sum_few_tiles(kSumF16KFirst, cus, m, n) || k > (tiles > cus ? 640 : 1023)) {
        const int32_t g = sum_groups_for(kSumF16KFirst, m, k, n, batch);
        return g == batch && batch > 1 ? 0 : g;
    }
    int32_t best = 0;
    float best_t = 1e30f;
    for (int32_t g = 1; g <= batch && (g == 1 || g * tiles <= 4 * cus); ++g) {
        if (batch % g != 0) continue;
        const float t = sum_krows_time(cus, tiles, m, k, n, batch, g);
        if (t < best_t) {
            best_t = t;
            best = g;
        }
    }
    return best;
}

static int32_t sum_groups_timed(int kind, int32_t m, int32_t k, int32_t n, int32_t batch) {
    if (kind == kSumF16KFirst) {
        const int32_t g = sum_krows_groups(m, k, n, batch);
        return g == 0 ? batch : g;
    }
    const int64_t cus = compute_units(), tiles = ceil_div(n, 128) * ceil_div(m, 128);
    if (!sum_few_tiles(kind, cus, m, n)) return sum_groups_for(kind, m, k, n, batch);
    int32_t best = batch;
    float best_t = sum_apart_time(kind == kSumI8, cus, tiles, m, k, n, batch);
    for (int32_t g = 1; g < batch && g * tiles <= 4 * cus; ++g) {
        if (batch % g != 0 || batch / g > kSumMax) continue;
        const float t = sum_group_time(kind == kSumI8, cus, tiles, m, k, n, batch, g);
        if (t < best_t) {
            best_t = t;
            best = g;
        }
    }
    return best;
}

// PART: fp32 out.  A group's sum may pass fp16's range where the sum over all groups does not: sums of more than one group stay
// fp32 until they are added up (cpmk_gemm_add_parts).
template <bool PART>
static int gemm_sum_dispatch(bool f16, int32_t m, int32_t k, int32_t n, int32_t batch, int32_t groups, const void* A, const void* B,
                             const void* srow, void* out, hipStream_t st) {
    constexpr int I8 = PART ? kEpiSumI8Part : kEpiSumI8, F16 = PART ? kEpiSumF16Part : kEpiSumF16;
    if (m < 0 || n < 0 || k <= 0 || batch < 1 || groups < 1 || batch % groups || batch / groups > kSumMax || groups > 65535) return CPMK_EBADARG;
    if (m % 4 || n % 4) return CPMK_EALIGN;
    if (m == 0 || n == 0) return 0;
    if (any_null(A, B, out) || (!f16 && srow == nullptr)) return CPMK_EBADARG;
    const int32_t kb = f16 ? 2 * k : k;        // bytes per row
    if (k > (1 << 29) || (int64_t)n * kb >= (1ll << 32) || (int64_t)m * kb >= (1ll << 32)) return CPMK_ETOOBIG;
    if (!aligned16(out) || (f16 ? (kb <= 64 || kb % 4 != 0) : kb % 128 != 0)) return CPMK_EALIGN;
    const bool whole = kb % 16 == 0 && aligned16(A) && aligned16(B);
    if (!whole && (!f16 || ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 3u))) return CPMK_EALIGN;
    GemmArgs a = {};
    a.P = (const int8_t*)B; a.Q = (const int8_t*)A; a.out = out;
    a.srow = (const half_t*)srow; a.scol = nullptr;
    a.strideP = (int64_t)n * kb;
    a.strideQ = (int64_t)m * kb;
    a.n = n; a.m = m; a.k = kb; a.bc_row = 0; a.bc_col = 0;
    a.tiles_r = a.tiles_c = 0;
    a.edge_in = 0;
    a.nsum = batch / groups;
    const uint32_t nkb = (uint32_t)(kb / (kb % 128 == 0 ? 128 : 64));
    if ((uint64_t)nkb * a.nsum >= 65536) return CPMK_ETOOBIG;
    a.kmagic = (uint32_t)(((1ull << 32) + nkb - 1) / nkb);
    const int64_t cus = compute_units();
    if (!f16) {
        // Bound by the LDS traffic of the K loop.  Beside the int32 accumulators a wave holds as many fp32 sums, so its share of
        // the tile is 64 x 64 where the plain product's is 128 x 64: 256x128 tiles of eight waves, whose fragment reads alone take as
        // long as their products (the DMA's writes come on top).  10240 x 4096 outputs over 8 entries of 512: 194 us (202 with an entry's
        // product folded between two slabs instead of under the next entry's first products), against 287 us for the products one by
        // one and 149 us for adding them up; waves of 128 x 64, one per SIMD, 316 us (their accumulators have to be carried
        // between the two register files to be folded).
        if (ceil_div(n, 256) * ceil_div(m, 128) * groups * 4 >= cus * 3) return launch_dma<4, 2, 2, 2, 128, I8, 2, 0, 16>(a, groups, st);
        // too few of them for most compute units: 128x128 tiles, two workgroups a compute unit when there are more than compute
        // units (1024 x 2560 over 4 x 256: 12.0 us; 15.2 as 256x128), else the deeper ring (2048 x 2048 over 8 x 512: 29.8 us; two stages 31.3)
        const int64_t mid = ceil_div(n, 128) * ceil_div(m, 128) * groups;
        if (mid > cus) return launch_dma<2, 2, 2, 2, 128, I8, 2, 0, 16>(a, groups, st, 2);
        return launch_dma<2, 2, 2, 2, 128, I8, kRingSmall, 0, 16>(a, groups, st);
    }
    const bool large = ceil_div(n, 256) * ceil_div(m, 256) * groups * 4 >= cus * 3;
    if (kb % 128 == 0) return large ? launch_dma<2, 4, 4, 2, 128, F16, 2, 0, 16>(a, groups, st) : launch_dma<2, 2, 2, 2, 128, F16, kRingSmall, 0, 16>(a, groups, st);
    if (whole) return large ? launch_dma<2, 4, 4, 2, 64, F16, 4, 4, 16>(a, groups, st) : launch_dma<2, 2, 2, 2, 64, F16, kRingSmall, 4, 16>(a, groups, st);
    return large ? launch_dma<2, 4, 4, 2, 64, F16, 4, 12, 16>(a, groups, st) : launch_dma<2, 2, 2, 2, 64, F16, kRingSmall, 12, 16>(a, groups, st);
}

// fp16 products whose operands are both stored (K, rows): the entries of a group lie one behind the other and are one
// contraction of `k` (all of them together) as they lie.  The tile kernel's part of gemm_f16_dispatch, fp32 out; `any`: what it does not take on the kernel for any size.
static int gemm_rows_parts(int32_t m, int64_t k, int32_t n, int32_t groups, const void* A, const void* B, void* out, bool any, hipStream_t st) {
    if (m < 0 || n < 0 || k < 0 || groups < 1) return CPMK_EBADARG;
    if (m % 2 || n % 2 || k % 2) return CPMK_EALIGN;
    if (m == 0 || n == 0) return 0;
    if (any_null(A, B, out)) return CPMK_EBADARG;
    if (n * k * 2 >= (1ll << 32) || m * k * 2 >= (1ll << 32)) return CPMK_ETOOBIG;
    const bool in_p = n % 8 != 0, in_q = m % 8 != 0;
    if (!aligned16(out)) return CPMK_EALIGN;
    if (!krows_tiles(m, k, n) || !aligned16(A) || !aligned16(B))
        return any ? gemm_f16_any(m, (int32_t)k, n, groups, groups, 0, 1, A, B, out, st, true) : CPMK_EALIGN;
    GemmArgs a = {};
    a.P = (const int8_t*)B; a.Q = (const int8_t*)A; a.out = out;
    a.srow = nullptr; a.scol = nullptr;
    a.strideP = n * k * 2;
    a.strideQ = m * k * 2;
    a.n = n; a.m = m; a.k = (int32_t)(k * 2); a.bc_row = 0; a.bc_col = 0;
    a.tiles_r = a.tiles_c = 0;
    a.edge_in = (in_p ? 1 : 0) | (in_q ? 2 : 0);
    a.nsum = 1;
    a.kmagic = 0;
    const int64_t big = ceil_div(n, 256) * ceil_div(m, 256), mid = ceil_div(n, 128) * ceil_div(m, 128);
    const bool large = big * 8 <= mid * 3 && big * groups * 4 >= (int64_t)compute_units() * 3 && n > 128 && m > 128 && (!in_p || n >= 256);
    const bool rest = k % 64 != 0;
    if (large) return rest ? launch_dma<2, 4, 4, 2, 128, kEpiF16Part, 2, 15, 16>(a, groups, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16Part, 2, 3, 16>(a, groups, st);
    return rest ? launch_dma<2, 2, 2, 2, 128, kEpiF16Part, 2, 15, 32>(a, groups, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16Part, kRingSmall, 3, 32>(a, groups, st);
}

// out[j] = fp16(sum over the groups of parts[g, j]), in the order of the groups.  Bound by reading the parts.  A lane owns four
// adjacent columns and requests eight groups at a time; with few columns the groups are dealt to `rgs` (a power of two up to 64)
// sets of 256 / rgs lanes, as in k_batch_add_backward.
__global__ __launch_bounds__(256) void k_add_parts(int32_t groups, int64_t n, int rgs, const float* __restrict__ parts, half_t* __restrict__ out) {
    __shared__ float red[1024];                 // [set][column of the workgroup]
    const int cgs = 256 / rgs, cg = threadIdx.x % cgs, rg = threadIdx.x / cgs;
    const int64_t col = ((int64_t)blockIdx.x * cgs + cg) * 4;
    const bool live = col < n;                  // (n % 4 == 0)
    float4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (live) {
        for (int32_t g0 = rg; g0 < groups; g0 += 8 * rgs) {
            float4_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int32_t g = g0 + u * rgs;
                v[u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                if (g < groups) v[u] = *reinterpret_cast<const float4_t*>(parts + g * n + col);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] += v[u][e];
        }
    }
    if (rgs > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) red[(rg * cgs + cg) * 4 + e] = s[e];
        __syncthreads();
        if (rg != 0) return;
        for (int g = 1; g < rgs; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += red[(g * cgs + cg) * 4 + e];
    }
    if (!live) return;
    half4_t r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (half_t)s[e];
    *reinterpret_cast<half4_t*>(out + col) = r;
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_gemm_sum_groups(int32_t m, int32_t n, int32_t batch) {
    return m < 0 || n < 0 || batch < 1 ? 1 : sum_groups(m, n, batch);
}

int cpmk_gemm_sum_groups_for(int kind, int32_t m, int32_t k, int32_t n, int32_t batch) {
    return m < 0 || n < 0 || k < 0 || batch < 1 ? 1 : sum_groups_for(kind, m, k, n, batch);
}

int cpmk_gemm_sum_groups_timed(int kind, int32_t m, int32_t k, int32_t n, int32_t batch) {
    return m <= 0 || n <= 0 || k <= 0 || batch < 1 ? 1 : sum_groups_timed(kind, m, k, n, batch);
}

int cpmk_gemm_sum_krows_groups(int32_t m, int32_t k, int32_t n, int32_t batch) {
    return m <= 0 || n <= 0 || k <= 0 || batch < 1 ? 0 : sum_krows_groups(m, k, n, batch);
}

int cpmk_gemm_int8_scale_sum(int32_t m, int32_t k, int32_t n, int32_t batch, int32_t groups, const void* A, const void* B,
                             const void* scale_row, void* out, void* stream) {
    clear_stale_error();
    return gemm_sum_dispatch<false>(false, m, k, n, batch, groups, A, B, scale_row, out, (hipStream_t)stream);
}

int cpmk_gemm_fp16_sum(int32_t m, int32_t k, int32_t n, int32_t batch, int32_t groups, const void* A, const void* B,
                       void* out, void* stream) {
    clear_stale_error();
    return gemm_sum_dispatch<false>(true, m, k, n, batch, groups, A, B, nullptr, out, (hipStream_t)stream);
}

int cpmk_gemm_int8_scale_parts(int32_t m, int32_t k, int32_t n, int32_t batch, int32_t groups, const void* A, const void* B,
                               const void* scale_row, void* parts, void* stream) {
    clear_stale_error();
    return gemm_sum_dispatch<true>(false, m, k, n, batch, groups, A, B, scale_row, parts, (hipStream_t)stream);
}

int cpmk_gemm_fp16_parts(int32_t m, int32_t k, int32_t n, int32_t batch, int32_t groups, int k_first, const void* A, const void* B,
                         void* parts, void* stream) {
    clear_stale_error();
    if (!k_first) return gemm_sum_dispatch<true>(true, m, k, n, batch, groups, A, B, nullptr, parts, (hipStream_t)stream);
    if (k < 0 || batch < 1 || groups < 1 || batch % groups) return CPMK_EBADARG;
    return gemm_rows_parts(m, (int64_t)k * (batch / groups), n, groups, A, B, parts, k_first == 2, (hipStream_t)stream);
}

int cpmk_gemm_add_parts(int32_t groups, int64_t n, const void* parts, void* out, void* stream) {
    clear_stale_error();
    if (groups < 1 || n < 0) return CPMK_EBADARG;
    if (n == 0) return 0;
    if (any_null(parts, out)) return CPMK_EBADARG;
    if (n % 4 || !aligned16(parts) || (reinterpret_cast<uintptr_t>(out) & 7u)) return CPMK_EALIGN;
    // enough lanes for the whole chip: with few columns, more sets of groups per workgroup
    int rgs = 1;
    while (rgs < 64 && n / 4 * rgs < 131072 && rgs * 2 <= groups) rgs *= 2;
    const int64_t blocks = ceil_div(n, 256 / rgs * 4);
    if (blocks >= 1 << 24) return CPMK_ETOOBIG;       // (a launch holds fewer than 2^32 threads)
    hipLaunchKernelGGL(k_add_parts, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, groups, n, rgs, (const float*)parts, (half_t*)out);
    return launch_status();
}

}  // extern "C"
