// Products whose depth is divided among workgroups: a product of few output tiles and a long contraction (a short prompt through a
// large projection, 120 x 3904 outputs over a depth of 12096) leaves most compute units idle, and those at work wait for one
// slab after the other.  Here a tile's depth is dealt to several workgroups, each of which stores its sums (exact int32, or fp32) in
// memory of the caller's, and a second kernel adds them up, dequantises and writes the result
// (cpm_kernels/torch/gemm.py:40-82, 189-203).
#include "gemm_tile.h"

namespace cpmk {

// What a product looks like to the kernels here, entries joined to one where they lie one behind the other.
struct PartsForm {
    int32_t n, m, entries;       // outputs of an entry, entries
    int32_t kb, slabs;           // bytes of the depth, 128-byte slabs
    int32_t seg;                 // columns of one caller's entry, where those are joined side by side, or 0
    bool pt, qt;                 // operands stored (K, rows)
    bool narrow;                 // tiles of 128 x 64 outputs, else 128 x 128
    int64_t tiles;               // of all entries
};

static bool parts_form(bool f16, int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, bool rows_ok, bool cols_ok, PartsForm& f) {
    const int32_t unit = f16 ? 8 : 16;       // elements of a 16-byte piece
    const int64_t batch = batchA > batchB ? batchA : batchB, kb = (int64_t)k * (f16 ? 2 : 1);
    f.pt = bT != 0;
    f.qt = aT == 0;
    if (kb % 128 != 0 || kb < 256 || kb >= 1 << 30 || m % 4 || n % 4 || (f.pt && n % unit) || (f.qt && (!f16 || m % unit))) return false;
    f.n = n; f.m = m; f.entries = (int32_t)batch; f.seg = 0;
    if (batch > 1 && batchA == 1 && !f.pt && rows_ok && rows_join((int)batch, n, kb)) {
        f.n = (int32_t)(n * batch);
        f.entries = 1;
    } else if (batch > 1 && batchB == 1 && !f.qt && cols_ok && cols_join((int)batch, m, kb)) {
        f.seg = m;
        f.m = (int32_t)(m * batch);
        f.entries = 1;
    }
    if (f.n * kb >= (1ll << 32) || f.m * kb >= (1ll << 32) || (int64_t)f.n * f.m * f.entries >= 1 << 28) return false;
    f.kb = (int32_t)kb;
    f.slabs = (int32_t)(kb / 128);
    f.narrow = f.m <= 64 && (f16 || !f.pt);        // (int8 operands stored (K, rows) are read in groups of 128 of their rows)
    f.tiles = ceil_div(f.n, 128) * ceil_div(f.m, f.narrow ? 64 : 128) * f.entries;
    return true;
}

struct AddPartsArgs {
    const void* parts;             // (parts, entries, n, m) int32 or fp32
    half_t* out;                   // (entries, n, m), or with seg (m / seg, n, seg)
    const half_t *srow, *scol;     // int8: scales as in GemmArgs
    int32_t bc_row, bc_col;
    int32_t count, n, m, seg;
    uint32_t total;                // entries * n * m
};

// Bound by reading the parts, which the products have just left in the caches.  A lane owns four adjacent columns and requests eight
// parts at a time.
template <bool I8>
__global__ __launch_bounds__(256) void k_add_depth_parts(AddPartsArgs a) {
    using vec_t = std::conditional_t<I8, int4_t, float4_t>;
    const uint32_t at = (blockIdx.x * 256u + threadIdx.x) * 4u;
    if (at >= a.total) return;
    const uint32_t row_all = at / (uint32_t)a.m, col = at - row_all * (uint32_t)a.m;         // m % 4 == 0
    const uint32_t e = row_all / (uint32_t)a.n, row = row_all - e * (uint32_t)a.n;
    const uint32_t ce = a.seg ? col / (uint32_t)a.seg : 0;
    half_t sxh = (half_t)1.0f;
    half4_t syh = {1, 1, 1, 1};
    if constexpr (I8) {
        if (a.srow) sxh = a.srow[a.bc_row ? row : row_all];
        if (a.scol) syh = *reinterpret_cast<const half4_t*>(a.scol + (a.bc_col || a.seg ? col : e * (uint32_t)a.m + col));
    }
    vec_t s = {0, 0, 0, 0};
    const vec_t* p = reinterpret_cast<const vec_t*>(a.parts) + at / 4;
    const uint32_t plane = a.total / 4;
    for (int32_t g0 = 0; g0 < a.count; g0 += 8) {
        vec_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            v[u] = vec_t{0, 0, 0, 0};
            if (g0 + u < a.count) v[u] = p[(int64_t)(g0 + u) * plane];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int c = 0; c < 4; ++c) s[c] += v[u][c];
    }
    half4_t r;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if constexpr (I8) r[c] = dequant(s[c], (float)sxh, (float)syh[c]);
        else r[c] = (half_t)s[c];
    }
    const int64_t o = a.seg ? ((int64_t)ce * a.n + row) * a.seg + (col - ce * (uint32_t)a.seg) : (int64_t)at;
    *reinterpret_cast<half4_t*>(a.out + o) = r;
}

template <int EPI, int LAY>
static int launch_parts(GemmArgs& a, int work, bool narrow, bool two, hipStream_t st) {
    if constexpr (EPI != kEpiInt32 || (LAY & 1) == 0)
        if (narrow) return two ? launch_dma<2, 2, 2, 1, 128, EPI, 2, LAY, 32>(a, work, st, 2) : launch_dma<2, 2, 2, 1, 128, EPI, kRingSmall, LAY, 32>(a, work, st);
    return two ? launch_dma<2, 2, 2, 2, 128, EPI, 2, LAY, 32>(a, work, st, 2) : launch_dma<2, 2, 2, 2, 128, EPI, kRingSmall, LAY, 32>(a, work, st);
}

static int parts_dispatch(bool f16, int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, const void* A, const void* B,
                          const void* srow, const void* scol, int bcr, int bcc, void* out, int32_t parts, void* ws, hipStream_t st) {
    if (m < 0 || n < 0 || k < 0 || batchA < 1 || batchB < 1 || parts < 1) return CPMK_EBADARG;
    if (!(batchA == batchB || batchA == 1 || batchB == 1)) return CPMK_EBADARG;
    if (m == 0 || n == 0) return 0;
    if (any_null(A, B, out) || ws == nullptr || (!f16 && srow == nullptr && scol == nullptr)) return CPMK_EBADARG;
    PartsForm f;
    if (!parts_form(f16, m, k, n, batchA, batchB, aT, bT, (srow == nullptr || !bcr) && (scol == nullptr || bcc), (srow == nullptr || bcr) && (scol == nullptr || !bcc), f)) return CPMK_EBADARG;
    if (!aligned16(A) || !aligned16(B) || !aligned16(ws) || (reinterpret_cast<uintptr_t>(out) & 7u) || (scol && (reinterpret_cast<uintptr_t>(scol) & 7u))) return CPMK_EALIGN;
    if (parts > f.slabs) parts = f.slabs;
    GemmArgs a = {};
    a.P = (const int8_t*)B; a.Q = (const int8_t*)A; a.out = ws;
    const bool joined = f.entries == 1;
    a.strideP = joined || batchB == 1 ? 0 : (int64_t)f.n * f.kb;
    a.strideQ = joined || batchA == 1 ? 0 : (int64_t)f.m * f.kb;
    a.n = f.n; a.m = f.m; a.k = f.kb;
    a.nsum = 1;
    a.entries = f.entries;
    a.part_slabs = (int32_t)ceil_div(f.slabs, parts);
    parts = (int32_t)ceil_div(f.slabs, a.part_slabs);       // (none without slabs)
    a.partP = (int64_t)a.part_slabs * 128 * (f.pt ? f.n : 1);
    a.partQ = (int64_t)a.part_slabs * 128 * (f.qt ? f.m : 1);
    const int64_t work = (int64_t)f.entries * parts, items = f.tiles * parts;
    if (work > 65535) return CPMK_ETOOBIG;
    const bool two = items > compute_units();
    const int lay = (f.pt ? 1 : 0) | (f.qt ? 2 : 0);
    int rc;
    if (!f16) rc = lay == 0 ? launch_parts<kEpiInt32, 32>(a, (int)work, f.narrow, two, st) : launch_parts<kEpiInt32, 33>(a, (int)work, f.narrow, two, st);
    else if (lay == 0) rc = launch_parts<kEpiF16Part, 32>(a, (int)work, f.narrow, two, st);
    else if (lay == 1) rc = launch_parts<kEpiF16Part, 33>(a, (int)work, f.narrow, two, st);
    else if (lay == 2) rc = launch_parts<kEpiF16Part, 34>(a, (int)work, f.narrow, two, st);
    else rc = launch_parts<kEpiF16Part, 35>(a, (int)work, f.narrow, two, st);
    if (rc != 0) return rc;
    AddPartsArgs p;
    p.parts = ws; p.out = (half_t*)out; p.srow = (const half_t*)srow; p.scol = (const half_t*)scol; p.bc_row = bcr; p.bc_col = bcc;
    p.count = parts; p.n = f.n; p.m = f.m; p.seg = f.seg;
    p.total = (uint32_t)((int64_t)f.entries * f.n * f.m);
    const dim3 grid((unsigned)ceil_div(p.total, 1024));
    if (f16) hipLaunchKernelGGL(k_add_depth_parts<false>, grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(k_add_depth_parts<true>, grid, dim3(256), 0, st, p);
    return launch_status();
}

// Parts to divide the depth of a product into, 1 where it is quicker whole.  In us, fitted to products of 8 to 230 tiles and depths of 4 to 151
// slabs, within 10 %: a slab of a tile takes 0.40 (fp16 0.44) with one workgroup a compute unit and 0.72 (0.80) with two, of a tile of 128 x 64
// outputs 0.31 (0.34), start and end of the product 4.5, the second kernel 3 and the time to write and read the parts at 4.7 TB/s.  Whole / divided:
// int8 120 x 3904, K = 4096 15.3 / 14.0 (3 parts, left whole), 8192 25.0 / 16.0 (6), 12160 34.3 / 18.3 (8); 136 x 3200 over 5 entries, K = 8192 39.5 / 33.2 (3);
// 512 x 4096, K = 12160 38.2 / 36.0 (2, left whole); fp16 56 x 4608, K = 1024 12.0 / 10.1 (left whole), 2048 19.1 / 11.6 (4), 9664 69 / 20.6 (6).
int32_t depth_parts(bool f16, int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, float* time) {
    PartsForm f;
    if (!parts_form(f16, m, k, n, batchA, batchB, aT, bT, true, true, f)) return 1;
    const int64_t cus = compute_units();
    const float one = f16 ? 0.44f : 0.40f, two = f16 ? 0.80f : 0.72f, thin = f16 ? 0.34f : 0.31f;
    const bool halves = !f16 && !f.pt && ceil_div(f.n, 128) * ceil_div(f.m, 64) * f.entries <= cus;      // (the whole product's tiles: gemm_dispatch)
    const float whole = 4.5f + (float)f.slabs * (halves ? thin : one);
    if (f.tiles >= cus) return 1;
    const float plane = 8e-6f * (float)f.n * (float)f.m * (float)f.entries / 4.7f;
    int32_t best = 1;
    float best_t = (whole - 2.0f) / 1.1f;        // (two kernels and a workspace cost the host too)
    for (int32_t s = 2; s <= 16 && s * 4 <= f.slabs && s * f.tiles <= 2 * cus; ++s) {
        const float slab = f.narrow ? (s * f.tiles <= cus ? thin : 2 * thin) : s * f.tiles <= cus ? one : two;
        const float t = 7.5f + (float)ceil_div(f.slabs, s) * slab + (float)s * plane;
        if (t < best_t) {
            best_t = t;
            best = s;
        }
    }
    if (best > 1 && time) *time = best_t;
    return best;
}

// fp16, a weight A (1, n, k) [(1, k, n) if aT] beside entries B (batch, k, m): estimates in us as above, of the product as it lies and with a copy of the
// entries as (batch, m, k), which are joined to one product then and whose depth may be divided, where entries stored (K, rows) of less than a
// tile, or of rows that are not whole 16-byte pieces, are a tile or more each, on the kernel for any size or on the tile kernel.  Fitted to 860 products of 4
// to 508 columns, 1 to 24 entries and depths of 256 to 24000 beside 128 to 10240 rows, the most within 15 %.
struct CopyTimes {
    float direct, copied;
};
static CopyTimes copy_times(int32_t n, int32_t k, int32_t m, int32_t batch, int aT) {
    const int64_t units = compute_units();
    const float cus = (float)units, slabs = (float)k / 64.0f, mb = 1e-6f * (float)k * (float)m * (float)batch;
    // (a round of large tiles, or tiles of 128 x 128 of up to a round, two, more of them; `apart`: of joined entries, big_tiles)
    auto tiled = [&](int64_t width, int64_t entries, int64_t apart, float base, float one, float two, float many, float large) {
        if (large > 0.0f && n > 128 && width > 128 && big_tiles(n, (int32_t)width, (int)entries, apart, units) * 4 >= units * 3)
            return (float)ceil_div(ceil_div(n, 256) * ceil_div(width, 256) * entries, units) * (slabs * large + 8.0f);
        const float rounds = (float)(ceil_div(n, 128) * ceil_div(width, 128) * entries) / cus;
        return base + slabs * (rounds <= 1.0f ? one : rounds <= 2.0f ? two : many * rounds);
    };
    const bool whole = k % 64 == 0;
    CopyTimes t;
    if (depth_parts(true, m, k, n, batch, 1, 0, aT, &t.direct) == 1) {
        if (m % 8 != 0 && m < 128) {
            const float rounds = (float)(ceil_div(n, 64) * ceil_div(m, 64) * batch) / cus;
            t.direct = 2.6f + slabs * (rounds <= 1.0f ? 0.58f : rounds <= 4.0f ? 1.1f : 0.29f * rounds);
        } else {
            const float large = m % 8 == 0 || m >= 256 ? 1.4f : 0.0f;
            t.direct = aT ? tiled(m, batch, 0, 4.8f, whole ? 0.49f : 0.58f, 0.8f, 0.86f, large) : whole ? tiled(m, batch, 0, 5.0f, 0.48f, 0.87f, 0.82f, large)
                                                                                                       : tiled(m, batch, 0, 7.7f, 0.46f, 1.24f, 0.92f, large);
        }
    }
    if (depth_parts(true, m, k, n, batch, 1, 1, aT, &t.copied) > 1) {
        t.copied += 3.0f + mb;
    } else {
        const int64_t apart = n > 128 && m > 128 ? ceil_div(n, 256) * ceil_div(m, 256) * batch : 0;
        const bool join = batch > 1 && (!aT || n % 8 == 0) && cols_join(batch, m, (int64_t)k * 2) && cols_join_pays_f16(n, m, k, aT, batch, apart);
        const int64_t width = join ? (int64_t)m * batch : m, entries = join ? 1 : batch, big = join ? apart : 0;
        t.copied = 2.0f * mb + (aT ? tiled(width, entries, big, 10.1f, 0.44f, 0.8f, 0.84f, 1.25f) : whole ? tiled(width, entries, big, 7.0f, 0.5f, 0.81f, 0.65f, 1.25f)
                                                                                                        : tiled(width, entries, big, 7.8f, 0.46f, 1.08f, 1.03f, 1.25f));
    }
    return t;
}

// Whether the copy pays (columns x entries x k beside rows, direct / with the copy, us: 24 x 1 x 4480 beside 1028 18.3 / 20.0; 12 x 5 x 1920 beside 3496 21 / 13;
// 108 x 1 x 640 beside 1452 7.8 / 12.2; 124 x 4 x 1152 beside 4224 26 / 19; 164 x 22 x 9344 beside 3072 392 / 225; 500 x 8 x 4096 beside 7996 220 / 223).  Over the 860 products the choice is 0.8 % behind
// the better form of each, always copying 16 %, never 16 %.  Rows of 4j + 2 columns stay as they are: they are not joined (81 products, 0.6 % behind).
static bool copy_pays(int32_t n, int32_t k, int32_t m, int32_t batch, int aT) {
    if (m >= 512 || m % 4 != 0 || k < 256 || n < 128 || (int64_t)m * batch * k >= 1ll << 30) return false;
    const CopyTimes t = copy_times(n, k, m, batch, aT);
    return t.copied < 0.95f * t.direct;
}

// The time of one product of two operands stored (K, rows), by the form that copy_pays and depth_parts choose
float krows_time(int32_t m, int32_t k, int32_t n) {
    const CopyTimes t = copy_times(n, k, m, 1, 1);
    return copy_pays(n, k, m, 1, 1) ? t.copied : t.direct;
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_gemm_depth_parts(int f16, int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT) {
    return m <= 0 || n <= 0 || k <= 0 || batchA < 1 || batchB < 1 ? 1 : depth_parts(f16 != 0, m, k, n, batchA, batchB, aT, bT);
}

int cpmk_gemm_fp16_copy_pays(int32_t m, int32_t k, int32_t n, int32_t batch, int bT) {
    return m > 0 && n > 0 && k > 0 && batch > 0 && copy_pays(n, k, m, batch, bT) ? 1 : 0;
}

int cpmk_gemm_int8_scale_split(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, const void* A, const void* B,
                               const void* scale_row, const void* scale_col, int broad_cast_row, int broad_cast_col, void* out, int32_t parts,
                               void* workspace, void* stream) {
    clear_stale_error();
    return parts_dispatch(false, m, k, n, batchA, batchB, aT, bT, A, B, scale_row, scale_col, broad_cast_row, broad_cast_col, out, parts, workspace,
                          (hipStream_t)stream);
}

int cpmk_gemm_fp16_split(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, const void* A, const void* B, void* out,
                         int32_t parts, void* workspace, void* stream) {
    clear_stale_error();
    return parts_dispatch(true, m, k, n, batchA, batchB, aT, bT, A, B, nullptr, nullptr, 0, 0, out, parts, workspace, (hipStream_t)stream);
}

}  // extern "C"
