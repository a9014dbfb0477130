// fp16 products with fp32 accumulation (cpm_kernels/kernels/gemm.py:188-256, cuBLASLt): which kernel takes which.  Operands P and Q as in
// gemm_i8.hip; the tile kernel of gemm_tile.h, kernels of their own for short depths (gemm_short.hip, gemm_rows.hip), few rows (gemm_low.hip) and
// everything else (gemm_any.hip).
#include "gemm_tile.h"

namespace cpmk {

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
    if (batchA == 1 && !bT && rows_join(batch, n, (int64_t)k * 2) && rows_join_pays_f16(n, m, k, aT, batch, big_apart)) {
        n *= batch;
        batch = batchB = 1;
    }
    // (columns: depths and buffers that the tile kernel takes beside a K-major Q)
    int32_t seg = 0;
    const uintptr_t operands = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B);
    if (batchB == 1 && aT && m % 4 == 0 && cols_join(batch, m, (int64_t)k * 2) && aligned16(out) && (int64_t)n * k * 2 < (1ll << 32) &&
        (bT ? k >= 64 && n % 8 == 0 && operands % 16 == 0 : k > 32 && operands % 4 == 0) &&
        cols_join_pays_f16(n, m, k, bT, batch, big_apart)) {
        seg = m;
        m *= batch;
        batch = batchA = 1;
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
    a.seg = seg;
    a.segmagic = seg ? (uint32_t)(((1ull << 32) + seg - 1) / seg) : 0;
    // The tile kernel stores 16-byte pieces of output rows that start on dwords, and 8-byte halves at a row's end.  Rows of 4j + 2
    // elements end in neither: their last column tile lies inside the matrix (edge_in), which takes a matrix of at least one tile.
    const bool odd = m % 4 != 0;
    // (The line at 192 columns was drawn for depths up to 128 with both operands stored (K, rows), which have a kernel of their own now; what it still keeps on
    // the general kernel is deeper or stored otherwise and would mostly be quicker on the tiles from 128 columns on: 80 of 150 x 150, both stored (K, rows),
    // K = 256 22.6 us and 8.6, K = 512 42.6 and 12.2; both K-major, K = 512 15.8 and 11.4, 300 of 130 x 130, K = 1000 84 and 103.)
    const bool wide = (reinterpret_cast<uintptr_t>(out) & 3u) == 0 && (!odd || m >= 192);
    const bool p_kmajor = !bT, q_kmajor = aT != 0;
    // A depth up to 128: kernels of their own, one for rows off cache lines where those are many (gemm_f16_rows), one of small tiles -- but where the output's
    // rows are not whole cache lines and it exceeds half of the last-level cache, the tile kernel, whose large tiles share fewer of the lines, unless those cover
    // much more than the matrix.  And the tile kernel too, beyond a quarter of that cache, where its large tiles cover no more than the small ones do, of which the last overlap the ones before
    // them: for depths of two slabs (7659 of 136 x 192, K = 128 217 us, 245 there; 976 of 200 x 1024 145 and 161; 5425 of 192 x 192 187 and 199), and
    // for an operand shared by the batch that is one large tile, of one whole slab or of two (2034 of 192 x 512 with the 192 shared, K = 64 104 and
    // 119; with the 512 shared 111 and 68; 976 of 400 x 512, the 400 shared, 106 and 71), or of two if it is the row operand (the same, K = 128, 134 and 146).
    if (!p_kmajor && !q_kmajor && k > 0 && k <= 128) {
        const int64_t big = ceil_div(n, 256) * ceil_div(m, 256), mid = ceil_div(n, 128) * ceil_div(m, 128), area = (int64_t)n * m, outs = batch * area;
        const bool large = big * 8 <= mid * 3 && big * batch * 4 >= (int64_t)compute_units() * 3;
        const bool exact = big * 4 == mid && (n % 8 == 0 || n >= 256) && (m % 8 == 0 || m >= 256) && wide && aligned16(A) && aligned16(B);
        const bool overlap = batchA == batchB ? k > 112 && mid * 65536 > 5 * area
                                              : mid * 131072 > 9 * area && (batchB == 1 ? k > 112 || (k == 64 && n <= 256) : m <= 256 && (k == 64 || k > 112));
        if (const int rc = gemm_f16_rows(m, k, n, batchA, batchB, A, B, out, st); rc >= 0) return rc;
        if (!large || ((m % 64 == 0 || outs <= 1 << 26) && !(exact && overlap && outs > 1 << 25)))
            if (const int rc = gemm_f16_short(m, k, n, batchA, batchB, A, B, out, st); rc >= 0) return rc;
    }
    if (p_kmajor && !q_kmajor && n <= 64 && k > 0)       // probabilities x values
        if (const int rc = gemm_f16_low(m, k, n, batchA, batchB, A, B, out, st); rc >= 0) return rc;
    // Few rows or columns: the tile kernel's workgroups are one or two a compute unit and its prologue and epilogue overlap nothing, so products that are not
    // deep, or have workgroups for every compute unit and more, go to the kernel of small workgroups (n x m x k over as many entries as
    // make the tiles given; us there and here).  Q K-major: 64 x 250 x 250, 500 tiles 12.0 / 9.6; 64 x 512 x 512, 500 18.7 / 14.3, 250 9.9 / 10.5; 64 x 1022 x 1022,
    // 1000 81 / 67; 80 x 512 x 512, 500 19.9 / 16.7; 80 x 904 x 904, 1000 51.5 / 57.8; 128 x 700 x 700, 3000 211 / 182.  Q stored (K, rows): 80 x 300 x 300, 500 17.5 / 13.9,
    // 250 12.7 / 9.0; 128 x 512 x 512, 500 23.4 / 18.8, 250 14.2 / 14.3; 96 x 904 x 904, 500 29.3 / 29.2; beside fewer than 128 columns 64 x 64 x 64, 100 5.5 / 4.0.
    // Both stored (K, rows): 64 x 64 x 64, 100 5.5 / 3.8.
    if (k > 0 && seg == 0) {
        const int64_t tiles = ceil_div(m, 128) * batch, many = (int64_t)compute_units() * 7 / 4;
        bool few = false;
        if (p_kmajor && q_kmajor)
            few = n <= 128 && (k <= 256 || (tiles >= many && (n <= 64 || (k % 64 == 0 ? k <= 512 : tiles >= 2000))));
        else if (p_kmajor)
            few = (n <= 128 && (n > 64 || m < 128) && (k <= 448 || (k <= 704 && tiles >= many)));
        else if (!q_kmajor)
            few = (n < 128 || m < 128) && k <= 256;
        if (few) return gemm_f16_any(m, k, n, batchA, batchB, aT, bT, A, B, out, st);
    }
    // (LAY bit 4: the columns of several entries)
    auto kmajor = [&](auto segc) __attribute__((always_inline)) {
        constexpr int SEG = decltype(segc)::value ? 16 : 0;
        const int64_t big = big_tiles(n, m, batch, big_apart);
        const bool large = big * 4 >= compute_units() * 3 && n > 128 && m > 128 && (!odd || m >= 256), pieces = operands % 16 == 0;
        a.edge_in = odd ? 2 : 0;
        // A depth that is whole 128-byte slabs, whole 64-byte ones (96, 160 ...) or neither: then the rest of it comes straight from memory into the fragments
        // (large tiles) or as a slab filled up with zeros, as whole pieces (LAY bit 2) or as dwords (bit 3 too).
        const bool whole64 = k % 32 == 0 && pieces, whole128 = whole64 && k % 64 == 0, rest16 = k % 8 == 0 && pieces;
        if (large) {
            if (whole128 && k >= 256) return launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, SEG, 16>(a, batch, st);
            // Rows off cache lines: a 64-byte piece of a row lies in two lines nearly as often as a 128-byte one, so the longer slabs ask for a third
            // fewer (2700 x 8000, k = 1000 79.6 -> 65.3 us, 1500 121.9 -> 95.3, 9196 652 -> 487; 500 52.2 and 54.3).
            if (!whole128 && k >= 704)
                return rest16 ? launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, SEG | 4, 16>(a, batch, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, SEG | 12, 16>(a, batch, st);
            // Products of a few slabs -- attention scores, K = 64 -- are all prologue and epilogue, bound by the stores:
            // the 32x32 form is quicker there, and waves of 64 rows x 128 columns, whose row segments are 256 bytes,
            // store 5-15 % faster than waves of 128 x 64 (slabs of 64 bytes make room for their wider output strips)
            if (whole64) return launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, SEG, 32>(a, batch, st);
            return rest16 ? launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, SEG | 4, 32>(a, batch, st) : launch_dma<4, 2, 2, 4, 64, kEpiF16, 2, SEG | 12, 32>(a, batch, st);
        }
        // (as for int8: more 128x128 tiles than compute units but at most two each -> two workgroups per compute unit)
        const int64_t mid = ceil_div(n, 128) * ceil_div(m, 128) * batch, cus = compute_units();
        const bool two = mid > cus && mid <= 2 * cus;
        if (whole128)
            return two ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, SEG, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, SEG, 32>(a, batch, st);
        // The same choice of slabs where rows are off cache lines: 1200 x 4004, 320 tiles, k = 200 11.6 us on 64-byte slabs, one workgroup a compute unit, 10.6 so with two and 11.0 on 128-byte ones,
        // 500 18.4, 16.2 and 16.1, 1500 42.5, 38.0 and 31.5; 640 x 640, k = 1000 11.0 and 13.0, 2056 17.1 and 20.2, 1200 x 1500, 1500 22.0 and 19.8, 9196 120 and 88; 3000 x 3000, 500
        // 27.3 and 27.0, 1500 62.1 and 55.8.  (Rows of whole 64-byte slabs: 3000 x 3000, 1504 41.7 and 47.5.)
        // (Those are operands in reach of L2, where the shorter slabs stay ahead at any depth: 64 x 64, 1452 12.9 and 15.5.  Out of memory the longer ones are ahead from
        // 500 on, 640 x 640, 1540 34.6 and 28.5.  One line serves both.)
        if (!whole64 && two && k >= 320)
            return rest16 ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, SEG | 4, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, SEG | 12, 32>(a, batch, st, 2);
        if (!whole64 && !two && k >= (mid > cus ? 448 : rest16 ? 2816 : 1280))
            return rest16 ? launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, SEG | 4, 32>(a, batch, st) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, SEG | 12, 32>(a, batch, st);
        const int per_cu = two && k < 704 ? 2 : 1;
        if (whole64) return launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, SEG, 32>(a, batch, st, per_cu);
        return rest16 ? launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, SEG | 4, 32>(a, batch, st, per_cu)
                      : launch_dma<2, 2, 2, 2, 64, kEpiF16, kRingSmall, SEG | 12, 32>(a, batch, st, per_cu);
    };
    if (p_kmajor && q_kmajor && wide && k > 0 && (k > 32 ? operands % 4 == 0 : k == 32 && operands % 16 == 0) && (int64_t)n * k * 2 < (1ll << 32) &&
        (int64_t)m * k * 2 < (1ll << 32))
        return seg ? kmajor(std::true_type{}) : kmajor(std::false_type{});
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
        if (seg) {       // (P stored (K, rows))
            if (large) return rest ? launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 29, 16>(a, batch, st) : launch_dma<2, 4, 4, 2, 128, kEpiF16, 2, 17, 16>(a, batch, st);
            return rest ? launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 29, 32>(a, batch, st)
                 : two ? launch_dma<2, 2, 2, 2, 128, kEpiF16, 2, 17, 32>(a, batch, st, 2) : launch_dma<2, 2, 2, 2, 128, kEpiF16, kRingSmall, 17, 32>(a, batch, st);
        }
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
    if (seg) return CPMK_EBADARG;       // (never: joined products are the tile kernel's; here they would be written as one matrix)
    return gemm_f16_any(m, k, n, batchA, batchB, aT, bT, A, B, out, st);
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_gemm_fp16(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT,
                   const void* A, const void* B, void* out, void* stream) {
    clear_stale_error();
    return gemm_f16_dispatch(m, k, n, batchA, batchB, aT, bT, A, B, out, (hipStream_t)stream);
}

}  // extern "C"
