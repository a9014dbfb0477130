// The tile kernel of the matrix products: persistent workgroups, operand slabs by LDS DMA, MFMA, results through an LDS
// strip.  gemm_i8.hip holds the products with one output per batch entry, gemm_sum.hip those summed over the batch.
#pragma once
#include "common.h"
#include <type_traits>

namespace cpmk {

struct GemmArgs {
    const int8_t* P;      // row operand
    const int8_t* Q;      // column operand
    void* out;            // int32 or fp16, (batch, n, m)
    const half_t* srow;   // fused epilogue: scale per output row j (null: one)
    const half_t* scol;   // fused epilogue: scale per output column i (null: one)
    int64_t strideP, strideQ;   // batch strides in bytes (0 = broadcast)
    int32_t n, m, k;
    int32_t bc_row, bc_col;
    int32_t tiles_r, tiles_c;
    int32_t edge_in;      // bit 0 / 1: the last row / column tile starts at n - BR / m - BC instead of reaching past the end
    int32_t nsum;         // kEpiSum*: consecutive batch entries that one output is the sum of
    uint32_t kmagic;      // kEpiSum*: ceil(2^32 / slabs of one entry)
    int32_t seg;          // LAY bit 4: columns of one entry (the m columns are those of several entries side by side)
    uint32_t segmagic;    // ... ceil(2^32 / seg)
    int32_t entries;      // LAY bit 5: batch entries (work entry s * entries + e is part s of the depth of entry e),
    int32_t part_slabs;   // ... slabs of a part (the last one may have fewer)
    int64_t partP, partQ; // ... and bytes from one part's operands to the next's
};

// ---------------------------------------------------------------------------------------
// Persistent LDS-DMA kernel
// ---------------------------------------------------------------------------------------
template <int X, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (X < N) {
        f(std::integral_constant<int, X>{});
        static_for<X + 1, N>(f);
    }
}

// What the tile kernel does with its accumulators.
constexpr int kEpiInt32 = 0;     // int8 product, int32 out
constexpr int kEpiDequant = 1;   // int8 product, fp16( (f32(acc) * s_row) * s_col ) out
constexpr int kEpiF16 = 2;       // fp16 product with fp32 accumulation, fp16 out
// Sums over groups of `nsum` batch entries (the gradient of an operand that the forward product broadcast over the
// batch): the K loop runs through the slabs of one entry after the other, so the products of the single entries never
// travel through memory.  Both operands K-major.
constexpr int kEpiSumI8 = 3;     // int8 products: fp32 sums of f32(acc) * s_row of each entry, fp16 out
constexpr int kEpiSumF16 = 4;    // fp16 products: one fp32 accumulation over all entries, fp16 out
// The same, and the fp16 product, with fp32 out: partial sums, which may pass fp16's range although the whole sum does not.
constexpr int kEpiSumI8Part = 5, kEpiSumF16Part = 6, kEpiF16Part = 7;
constexpr bool epi_part(int e) { return e == kEpiSumI8Part || e == kEpiSumF16Part || e == kEpiF16Part; }
constexpr bool epi_fold(int e) { return e == kEpiSumI8 || e == kEpiSumI8Part; }
constexpr bool epi_f16(int e) { return e == kEpiF16 || e == kEpiF16Part || e == kEpiSumF16 || e == kEpiSumF16Part; }
constexpr bool epi_sum(int e) { return epi_fold(e) || e == kEpiSumF16 || e == kEpiSumF16Part; }
constexpr bool epi_out32(int e) { return e == kEpiInt32 || epi_part(e); }      // four bytes per output

struct DmaArgs {
    GemmArgs g;
    int32_t batch;
    int32_t ntiles;    // full-size tiles per batch entry (tiles_r x tiles_c)
    uint32_t nfull;    // work items [0, nfull) are whole tiles in walk order ...
    uint32_t nhalf;    // ... items [nfull, nfull + nhalf) are row halves (top, bottom) of the tiles that follow
};

// One work item of the persistent kernel: a whole BR x BC tile, or its top/bottom half.
struct GemmItem {
    uint32_t b;        // batch entry
    int32_t j0, i0;    // first output row / column
    bool half;
    bool valid;
};

// Tiles are walked in groups of GRP row tiles, column-major inside a group, so neighbours in the
// walk share operand slabs in L2.
template <int BR, int BC>
__device__ __forceinline__ GemmItem gemm_item(uint32_t L, const DmaArgs& da) {
    GemmItem it;
    it.valid = L < da.nfull + da.nhalf;
    it.half = L >= da.nfull;
    const uint32_t h = it.half ? L - da.nfull : 0;
    const uint32_t id = it.half ? da.nfull + (h >> 1) : L;
    it.b = id / (uint32_t)da.ntiles;
    const uint32_t t = id - it.b * (uint32_t)da.ntiles;
    constexpr uint32_t GRP = 4;
    const uint32_t group_sz = GRP * (uint32_t)da.g.tiles_c;
    const uint32_t g = t / group_sz;
    const uint32_t rows_in_group = min(GRP, (uint32_t)da.g.tiles_r - g * GRP);
    const uint32_t tin = t - g * group_sz;
    it.j0 = (int32_t)((g * GRP + tin % rows_in_group) * BR + (h & 1) * (BR / 2));
    it.i0 = (int32_t)((tin / rows_in_group) * BC);
    // An operand stored (K, rows) whose rows are not whole 16-byte pieces cannot be read past the matrix's edge piece by
    // piece, and output rows of 4j + 2 elements end in less than half a piece: the last tile then lies inside the matrix and
    // overlaps its neighbour, whose outputs it computes again (the same bits, stored twice).
    if (da.g.edge_in & 1) it.j0 = min(it.j0, da.g.n - BR);
    if (da.g.edge_in & 2) it.i0 = min(it.i0, da.g.m - BC);
    return it;
}

// A 16-byte piece of an output row on its way to memory; `left` = elements from the piece's first to the end of
// the row (a multiple of 4, at least 4; at least 8 in a tile that lies inside the matrix, see edge_in).  fp16 rows of 8j + 4 elements start on 8-byte boundaries and end in half a piece:
// whole pieces leave as 16 bytes wherever they lie (global stores need no alignment; as two 8-byte halves the scores of 1024 heads
// of 500 x 500 took 175 us instead of 163, 128 heads of 588 x 588 52 instead of 46).
template <int ESZ>
__device__ __forceinline__ void store_piece(int8_t* dst, int4_t v, int32_t left) {
    struct __attribute__((packed, aligned(4))) Int4Any { int32_t x, y, z, w; };
    if (ESZ == 4 || left >= 8) {
        *reinterpret_cast<Int4Any*>(dst) = Int4Any{v.x, v.y, v.z, v.w};      // (the non-temporal hint changes nothing here: 133.7 against 134.1-135.2 us)
    } else {
        *reinterpret_cast<int2_t*>(dst) = int2_t{v.x, v.y};
    }
}

// What the two forms of the tile function below share: the rows a wave's DMA instructions fetch, a slab's place in
// the ring, what the last iterations of a tile fetch (the "tail"), and the priming of the ring at a tile's start.
// BR x BC outputs per workgroup of NW waves, BKB bytes of K per slab, NST ring stages; LAY / F16 as in the tile functions.
// TSW: a (K, L) operand lands with the units of every row of K exchanged within their 128-byte group -- fp16: unit
// (32 bytes) u of row k at u ^ (k & 3); int8: unit (16 bytes) u at u ^ (k & 7) -- which is what keeps the transposing
// fragment reads free of bank conflicts.  The DMA writes LDS in lane order, so the exchange happens in the choice of
// what a lane fetches.
// SUM: slab kt of a tile is slab kt % nkb of batch entry kt / nkb (counted from the tile's first entry).
// REST: a depth that is not whole slabs has the rest of it (`rem` bytes of a K-major row, any number of dwords) as slab 0
// and its whole slabs behind that one.  What the DMA fetches past the end of K -- the last 16 bytes of a K-major row, the
// last row of a (K, L) operand, again and again -- each lane puts right in LDS once slab 0 has landed (finish_rest): dwords
// moved down to their places, zeros beyond K.
template <int BR, int BC, int BKB, int NW, int NST, int LAY, bool F16, bool TSW = false, bool SUM = false, bool REST = false>
struct SlabDma {
    static_assert(!(REST && SUM), "sums over the batch take the rest of the depth from memory");
    static constexpr bool PARTS = (LAY & 32) != 0;        // the work entry is one part of the depth of its batch entry
    static_assert(!(PARTS && (REST || SUM)), "parts of the depth are whole slabs");
    static constexpr bool PT = (LAY & 1) != 0, QT = (LAY & 2) != 0;
    static constexpr int ESZ_IN = F16 ? 2 : 1;            // bytes per operand element
    static constexpr int EPP = 16 / ESZ_IN;               // elements per 16-byte piece
    static constexpr int CPR = BKB / 16;                  // 16-byte chunks per row of a slab
    static constexpr int RPW = 256 / BKB;                 // rows per 256-byte bank wrap
    static constexpr int STAGE = (BR + BC) * BKB;
    static constexpr int RPI = 1024 / BKB;                // rows per DMA instruction
    static constexpr int NDMA = (BR + BC) / RPI;
    static_assert(NDMA % NW == 0, "stage must split evenly over the waves");
    static_assert(!TSW || ((BR * ESZ_IN) % 128 == 0 && (BC * ESZ_IN) % 128 == 0), "the exchange of units stays inside whole 128-byte groups of a row of K");
    static constexpr int CNT = NDMA / NW;                 // DMA instructions per wave and slab

    const GemmArgs& a;
    const int wave, lane;
    int nk;                     // slabs per tile
    int nkb;                    // ... and per batch entry
    int rem;                    // REST: bytes of K in slab 0, or 0: whole slabs only
    int first;                  // slabs from the bases to the operands' starts
    int32_t oj0, oi0;           // first row / column of the tile
    bool ahead;                 // the next tile is fetched ahead (only if its LDS layout is this one's)
    bool deep;                  // at least as many slabs as stages
    int LD;                     // slabs in flight: the slab requested at iteration `it` is number it + LD of this tile
    int ring0;                  // stage of this tile's slab 0
    int32_t tj0, ti0;           // rows / columns the tail fetches
    const int8_t *Pb, *Qb, *Pn, *Qn;
    const int8_t *Pk, *Qk;      // SUM: the slab requested next,
    int left, step;             // ... slabs up to its entry's end and bytes to the next
    uint32_t voff[CNT], ldst[CNT];
    bool isq[CNT];
    int64_t kstepP, kstepQ;     // bytes from one K slab to the next

    __device__ __forceinline__ static int swz(int r) { return (r / RPW) & (CPR - 1); }

    // byte offset of this lane's 16 bytes inside slab 0 of the tile at rows oj / columns oi, for the wave's DMA
    // instruction d -> stage rows [RPI*dd, RPI*dd + RPI), dd = wave + d*NW; rows past the matrix are clamped (they only
    // feed outputs that are never stored)
    __device__ __forceinline__ uint32_t calc_voff(int d, int32_t oj, int32_t oi) const {
        const int dd = wave + d * NW;
        const int r = dd * RPI + lane / CPR;
        const int c = (lane % CPR) ^ swz(r);
        const bool q = dd * RPI >= BR;
        if ((PT && !q) || (QT && q)) {
            // a (K, L) operand: the instruction covers 1024 / (2 * B) rows of K, a lane one 16-byte piece of a row
            const int ppr = (q ? BC : BR) / EPP;                   // pieces per row of K
            const int dl = q ? dd - BR / RPI : dd;
            const int kr = dl * (64 / ppr) + lane / ppr;
            const int pl = lane % ppr;                             // the piece's place in the row of K in LDS
            const int pc = !TSW ? pl : F16 ? ((((pl >> 1) ^ (kr & 3)) << 1) | (pl & 1)) : (pl ^ (kr & 7));      // ... and which piece of the row it is
            const int32_t L = q ? a.m : a.n;
            return ((uint32_t)kr * (uint32_t)L + (uint32_t)min((q ? oi : oj) + pc * EPP, L - EPP)) * (uint32_t)ESZ_IN;      // L % EPP == 0
        }
        const int32_t grow = q ? min(oi + (r - BR), a.m - 1) : min(oj + r, a.n - 1);
        return (uint32_t)grow * (uint32_t)a.k + c * 16;
    }

    // REST: the same for slab 0, counted from the operand's start (operands are below 4 GiB)
    __device__ __forceinline__ uint32_t rest_voff(int d, int32_t oj, int32_t oi) const {
        const int dd = wave + d * NW;
        const bool q = dd * RPI >= BR;
        if ((PT && !q) || (QT && q)) {
            const int ppr = (q ? BC : BR) / EPP;
            const int kr = (q ? dd - BR / RPI : dd) * (64 / ppr) + lane / ppr;
            const int32_t L = q ? a.m : a.n;
            return calc_voff(d, oj, oi) + (uint32_t)((nk - 1) * (BKB / ESZ_IN) + min(kr, rem / ESZ_IN - 1) - kr) * (uint32_t)L * (uint32_t)ESZ_IN;
        }
        const int r = dd * RPI + lane / CPR;
        const int c = (lane % CPR) ^ swz(r);
        const int32_t grow = q ? min(oi + (r - BR), a.m - 1) : min(oj + r, a.n - 1);
        return (uint32_t)grow * (uint32_t)a.k + (uint32_t)((nk - 1) * BKB + min(c * 16, rem - 16));
    }

    __device__ __forceinline__ SlabDma(const GemmArgs& a_, uint32_t lds_base, const GemmItem& cur_item, const GemmItem& nxt_item,
                                       int wave_, int lane_, int ring)
        : a(a_), wave(wave_), lane(lane_) {
        nkb = a.k / BKB;
        rem = REST ? a.k - nkb * BKB : 0;
        nk = SUM ? nkb * a.nsum : REST && rem != 0 ? nkb + 1 : nkb;
        oj0 = cur_item.j0;
        oi0 = cur_item.i0;
        uint32_t b = SUM ? cur_item.b * (uint32_t)a.nsum : cur_item.b;
        uint32_t part = 0;
        if constexpr (PARTS) {
            part = b / (uint32_t)a.entries;
            b -= part * (uint32_t)a.entries;
            nk = nkb = min(a.part_slabs, nkb - (int)part * a.part_slabs);
        }
        Pb = a.P + (int64_t)b * a.strideP + (PARTS ? part * a.partP : 0);
        Qb = a.Q + (int64_t)b * a.strideQ + (PARTS ? part * a.partQ : 0);
        // (parts differ in their slabs: each is begun anew, as half tiles are.  The number of parts that the host picks leaves at most a tile a workgroup;
        // a caller's own may leave several.)
        ahead = !PARTS && nxt_item.valid && nxt_item.half == cur_item.half;
        // slab s of this tile lives in stage (ring + s) % NST.  With fewer slabs than stages (!deep) all of a
        // tile's slabs are requested one tile ahead and every wait is a full one.
        deep = nk >= NST;
        LD = deep ? NST : nk;
        ring0 = __builtin_amdgcn_readfirstlane(ring);
        // what the last LD iterations fetch: the next tile's first slabs, or (not ahead) this tile's last slab again
        const uint32_t tb = !ahead ? b : SUM ? nxt_item.b * (uint32_t)a.nsum : nxt_item.b;
        tj0 = ahead ? nxt_item.j0 : cur_item.j0;
        ti0 = ahead ? nxt_item.i0 : cur_item.i0;
        Pn = PARTS ? Pb : a.P + (int64_t)tb * a.strideP;
        Qn = PARTS ? Qb : a.Q + (int64_t)tb * a.strideQ;
#pragma unroll
        for (int d = 0; d < CNT; ++d) {
            const int dd = wave + d * NW;
            isq[d] = dd * RPI >= BR;
            voff[d] = calc_voff(d, cur_item.j0, cur_item.i0);
            ldst[d] = lds_base + dd * 1024;
        }
        kstepP = PT ? (int64_t)BKB * a.n : BKB;
        kstepQ = QT ? (int64_t)BKB * a.m : BKB;
        // With the rest of the depth as slab 0 slab kt >= 1 is whole slab kt - 1.  The bases move, so that the K loop finds it at kt slabs
        // all the same: chosen there, slab by slab, the offset cost a fifth of the loop (512 x 140 products of depth 9616 77 -> 92 us).
        // Slab 0 is at `first` slabs, with the offsets of rest_voff.
        first = 0;
        if constexpr (REST) {
            if (rem != 0) {
                first = 1;
                Pb -= kstepP; Pn -= kstepP;
                Qb -= kstepQ; Qn -= kstepQ;
            }
        }
    }

    // One DMA instruction of slab kt into ring stage `stage`: of this tile's rows, or (TAIL) of the rows the last LD
    // iterations fetch -- the next tile's when it is fetched ahead, else this tile's again.  Which one is a
    // compile-time choice: a run-time select here makes the compiler branch inside the K loop, which splits its
    // body and breaks the MFMA/memory interleave.
    template <int d, bool TAIL>
    __device__ __forceinline__ void issue(int kt, int stage) const {
        // read every candidate first and select values, never addresses of the members
        const int8_t *pb = TAIL ? Pn : Pb, *qb = TAIL ? Qn : Qb;
        const uint32_t v = voff[d];            // (rewritten for the tail between the two loops: retarget)
        const bool q = isq[d];
        if constexpr (SUM) {
            lds_dma16(v, q ? Qk : Pk, ldst[d] + stage * STAGE);
        } else {
            lds_dma16(v, (q ? qb : pb) + kt * (q ? kstepQ : kstepP), ldst[d] + stage * STAGE);
        }
    }

    // SUM: the slab that issue() requests next, followed through the entries by one addition a slab: divided and multiplied out
    // request by request it held the K loop up (fp16, 1024 x 4096 outputs
    // over 8 x 1024: 108 -> 95 us; int8 43 -> 36 with its sum in 128x128 tiles, 8192 x 1024 over 7 x 1024 68 -> 62 us).
    // `tail`: of the next tile, or (not ahead) this tile's last slab again and again.
    __device__ __forceinline__ void seek(bool tail, int kt) {
        const uint32_t e = nkb == 1 ? (uint32_t)kt : __umulhi((uint32_t)kt, a.kmagic);       // kt / nkb (exact for kt * nkb < 2^32)
        left = nkb - (kt - (int)e * nkb);
        const int32_t in_entry = (nkb - left) * BKB;
        Pk = (tail ? Pn : Pb) + ((int64_t)e * a.strideP + in_entry);
        Qk = (tail ? Qn : Qb) + ((int64_t)e * a.strideQ + in_entry);
        step = BKB;
        if (tail && !ahead) {
            step = 0;
            left = 0;
        }
    }
    __device__ __forceinline__ void advance() {
        const bool wrap = --left == 0;
        Pk += step + (wrap ? a.strideP - nkb * BKB : 0);
        Qk += step + (wrap ? a.strideQ - nkb * BKB : 0);
        left = wrap ? nkb : left;
    }

    // between a tile's main iterations and its tail: the offsets of the rows the tail fetches
    __device__ __forceinline__ void retarget() {
#pragma unroll
        for (int d = 0; d < CNT; ++d) voff[d] = calc_voff(d, tj0, ti0);
    }
    // ... and those of their slab 0, where that is the rest of the depth
    __device__ __forceinline__ void retarget_rest() {
#pragma unroll
        for (int d = 0; d < CNT; ++d) voff[d] = rest_voff(d, tj0, ti0);
    }

    // Slab 0 as the DMA left it -> the rest of the depth followed by zeros.  Every lane works on the 16 bytes it fetched itself, so
    // its own wave's wait before and the workgroup's barrier after are all it takes.
    __device__ __forceinline__ void finish_rest() const {
        if (rem == 0) return;
        typedef __attribute__((address_space(3))) int4_t* lds_ptr;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < CNT; ++d) {
            const int dd = wave + d * NW;
            const bool q = isq[d];
            lds_ptr p = (lds_ptr)(uintptr_t)(ldst[d] + (uint32_t)(ring0 * STAGE + lane * 16));
            if ((PT && !q) || (QT && q)) {
                const int ppr = (q ? BC : BR) / EPP;
                const int kr = (q ? dd - BR / RPI : dd) * (64 / ppr) + lane / ppr;
                if (kr * ESZ_IN >= rem) *p = int4_t{0, 0, 0, 0};
            } else {
                const int c = (lane % CPR) ^ swz(dd * RPI + lane / CPR);
                const int over = min(c * 16 + 16 - rem, 16);       // bytes of the piece beyond K: 4 ... 16 (or none)
                if (over > 0) {
                    const int4_t t = *p;
                    const int32_t w[8] = {t.x, t.y, t.z, t.w, 0, 0, 0, 0};
                    const int sh = over >> 2;
                    int4_t v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = sh == 1 ? w[e + 1] : sh == 2 ? w[e + 2] : sh == 3 ? w[e + 3] : 0;
                    *p = v;
                }
            }
        }
        asm volatile("" ::: "memory");
    }

    // A tile's start.  Without slabs on their way: request the first NST, wait for slab 0.  Otherwise the first LD
    // slabs were requested during the previous tile; its stores drain too.
    __device__ __forceinline__ void prime(bool have_slabs) {
        if (!have_slabs) {
            __syncthreads();                 // every wave is done with the ring of the previous tile
            static_for<0, NST>([&](auto sc) __attribute__((always_inline)) {
                constexpr int st = decltype(sc)::value;
                static_for<0, CNT>([&](auto dc) __attribute__((always_inline)) {
                    constexpr int d = decltype(dc)::value;
                    if constexpr (REST && st == 0) {
                        if (rem != 0) {
                            lds_dma16(rest_voff(d, oj0, oi0), (isq[d] ? Qb + kstepQ : Pb + kstepP), ldst[d] + ring0 * STAGE);
                            return;
                        }
                    }
                    if constexpr (SUM && d == 0) seek(false, min(st, nk - 1));
                    issue<d, false>(min(st, nk - 1), (ring0 + st) % NST);
                });
            });
            if (deep) wait_vmcnt<(NST - 1) * CNT>();   // slab 0 (and the scale loads issued before it) has landed
            else wait_vmcnt<0>();
            if constexpr (REST) finish_rest();
            __syncthreads();
        } else {
            wait_vmcnt<0>();
            if constexpr (REST) finish_rest();
            __syncthreads();
        }
    }
};

// The last iterations of a tile, from `it` on: the next tile's slab 0 first, which has offsets of its own where it is the rest of
// the depth.
template <bool REST, class Dma, class F>
__device__ __forceinline__ void tail_slabs(Dma& dma, int it, F&& slab) {
    if constexpr (REST) {
        const int first = it;
        for (; it < dma.nk; ++it) {
            if (it == first && dma.ahead && dma.rem != 0) dma.retarget_rest();
            else if (it <= first + 1) dma.retarget();
            slab(it, std::true_type{});
        }
    } else {
        dma.retarget();
        for (; it < dma.nk; ++it) slab(it, std::true_type{});
    }
}

// The way out of a tile, shared by the two forms of the tile function.  Results leave through a 4 KB strip of
// LDS per wave: a lane holds 4-column pieces of ONE output row, so storing straight from the accumulators
// would touch 32 different rows with 8 or 16 bytes each per instruction.  Written to the strip as 32 rows x RB
// bytes and read back 16 bytes per lane, every store instruction covers whole contiguous rows of the chunk
// (RB = 128 bytes: eight lanes per 128-byte line).
// SEG: the columns are those of several entries side by side, `a.seg` (a multiple of 4) each, and go out to one (n, seg) matrix an entry.
template <int EPI, int TC, bool SEG = false>
struct StripOut {
    static constexpr int ESZ = epi_out32(EPI) ? 4 : 2;
    static constexpr int CT = epi_out32(EPI) ? 1 : TC;       // MFMA tile columns (of 32) side by side in one chunk
    static constexpr int NCH = epi_out32(EPI) ? TC : 1;      // chunks per block of 32 rows
    static constexpr int RB = CT * 32 * ESZ, PPR = RB / 16, RPW2 = 256 / RB, PASSES = PPR / 2, RPP = 64 / PPR;
    // 16-byte piece p of strip row r sits at piece slot p ^ ((r / RPW2) % PPR): reads are conflict free
    static __device__ __forceinline__ int slot(int r, int p) { return (p ^ ((r / RPW2) & (PPR - 1))) << 4; }
    // the strip's 32 rows go out: output rows row0 .. row0 + 31, columns from col0 on
    static __device__ __forceinline__ void store_rows(const GemmArgs& a, const int8_t* stg, int64_t obase, int32_t row0, int32_t col0, int lane) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ++ps) {
            const int R = ps * RPP + lane / PPR, pc = lane % PPR;
            const int4_t v = *reinterpret_cast<const int4_t*>(stg + R * RB + slot(R, pc));
            const int32_t row = row0 + R;
            const int32_t col = col0 + pc * (16 / ESZ);
            if constexpr (SEG) {
                static_assert(ESZ == 2, "fp16 results");
                if (row < a.n && col < a.m) {
                    const uint32_t e = __umulhi((uint32_t)col, a.segmagic);          // col / seg (exact for m * seg < 2^32)
                    const int32_t c = col - (int32_t)e * a.seg;
                    half_t* dst = reinterpret_cast<half_t*>(a.out) + ((int64_t)e * a.n + row) * a.seg + c;
                    store_piece<ESZ>(reinterpret_cast<int8_t*>(dst), v, a.seg - c);
                    if (a.seg - c < 8 && col + 4 < a.m)      // the piece's second half is the next entry's
                        *reinterpret_cast<int2_t*>(reinterpret_cast<half_t*>(a.out) + ((int64_t)(e + 1) * a.n + row) * a.seg) = int2_t{v.z, v.w};
                }
            } else if (row < a.n && col < a.m)
                store_piece<ESZ>(reinterpret_cast<int8_t*>(a.out) + (obase + (int64_t)row * a.m + col) * ESZ, v, a.m - col);
        }
    }
};

// One output tile of BR x BC = (WR*TR*32) x (WC*TC*32), K slab = BKB bytes.
// The MFMA is the 16x16 one with 64 bytes of K (v_mfma_i32_16x16x64_i8, v_mfma_f32_16x16x32_f16):
// per operation it moves half the accumulator registers of the 32x32 form, and on random operands,
// where the chip's power limit sets the clock, the same product finishes about a tenth sooner.
// A wave owns AR x AC = 2TR x 2TC such tiles; lane (r = l % 16, q = l / 16) feeds 16 bytes of K
// (chunk q of the k-step) of row r of each operand block and receives output row r, columns
// 4q .. 4q+3 of each 16x16 tile (the operands are passed swapped).
// A k-step is two passes over the wave's rows, one per half of its columns: the column fragments
// come in two sets, one multiplied while the other is read, and a row fragment's register is
// refilled with the next k-step's right after its last MFMA of the second pass.
// NST-stage ring; pipeline per K slab `it` (stage cur = it % NST, slabs it+1 .. it+NST-1 in flight):
//   k-steps 0 .. KS-2, and the first pass of k-step KS-1 : MFMAs while the fragments that come
//                       next are read from stage cur
//   s_waitcnt vmcnt((NST-2)*CNT); barrier -> slab it+1 has landed in stage nxt for every wave and
//                                      nobody reads stage cur any more
//   second pass of k-step KS-1 : MFMAs while the step-0 fragments of slab it+1 are read and
//                       the DMA of slab it+NST is issued into stage cur
// The last iterations (the "tail", a second copy of the loop body) fetch the first slabs of the
// NEXT tile of this workgroup when it has the same shape, so that tile starts with its operands
// already in LDS and the loads overlap this tile's stores; otherwise they fetch this tile's last
// slab again (a redundant load nobody reads).  The ring position carries over from tile to tile
// (`ring`), so any slab count works.  Each loop body is one basic block without selects, which
// lets the compiler keep the accumulators in place and the MFMA/memory interleave as written.
// Returns true if the next tile's first slabs are on their way.
//
// LAY bit 2: the depth is not whole slabs (any multiple of 4 bytes).  Here the slabs of the ring cover the whole ones; the
// rest of the depth (less than a slab) goes from memory straight into the fragment registers before the K loop starts
// -- a lane's 16 bytes of a k-step are the same bytes in memory as in the stage -- with zeros past the end of K.  (Beside an
// operand stored (K, rows) the rest is a slab of the ring: SlabDma's REST.)
// LAY bit 3, with bit 2: the rest of a row may start off a 16-byte boundary and end inside a piece (depths and rows of
// whole dwords only); without it every piece of the rest is whole and aligned.
// LAY bit 4: the columns of several batch entries side by side (StripOut's SEG).  LAY bit 5: an entry's depth in parts, each a
// work entry with an output of its own (SlabDma's PARTS).
// LAY marks operands whose rows are K instead: bit 0 = the row operand is stored (K, n), bit 1 =
// the column operand is stored (K, m).  Such an operand's part of a stage holds the slab's rows
// of K (64 for fp16, 128 for int8) with the tile's BR (BC) elements each, DMA'd as they lie in
// memory (with the units of a row exchanged, SlabDma's TSW); a lane then gets its 16 bytes of K with two
// transposing LDS reads instead of one 16-byte read.
template <int WR, int WC, int TR, int TC, int BKB, int EPI, int NST, int LAY = 0>
__device__ __forceinline__ bool gemm_dma_tile(const GemmArgs& a, int8_t* smem, int8_t* stg, uint32_t lds_base,
                                              const GemmItem cur_item, const GemmItem nxt_item, const bool have_slabs, int& ring) {
    constexpr bool FUSED = EPI == kEpiDequant, F16 = epi_f16(EPI);
    constexpr bool SUM = epi_sum(EPI), FOLD = epi_fold(EPI);
    static_assert(!SUM || (LAY & 3) == 0, "sums over the batch: K-major operands");
    constexpr bool PT = (LAY & 1) != 0, QT = (LAY & 2) != 0;
    static_assert((LAY & 3) == 0 || BKB == 128, "transposed operands: 128 bytes of K per slab");
    constexpr int ESZ_IN = F16 ? 2 : 1;            // bytes per operand element
    using acc_t = std::conditional_t<F16, float4_t, int4_t>;
    constexpr int KS = BKB / 64, CPR = BKB / 16;
    static_assert(KS >= 1, "k-steps of 64 bytes");
    constexpr int AR = TR * 2, AC = TC * 2;        // 16x16 MFMA tiles of a wave
    constexpr int NW = WR * WC, BR = WR * TR * 32, BC = WC * TC * 32;
    constexpr bool TRP = PT, TRQ = QT;             // fragments of a (K, L) operand: transposing LDS reads
    constexpr bool REST = (LAY & 4) != 0 && (PT || QT);       // the rest of the depth is a slab of the ring
    using Dma = SlabDma<BR, BC, BKB, NW, NST, LAY, F16, TRP || TRQ, SUM, REST>;
    constexpr int STAGE = Dma::STAGE, CNT = Dma::CNT;      // bytes per ring stage; DMA instructions per wave and slab
    constexpr int RPW = 256 / BKB;                 // rows per 256-byte bank wrap
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC;
    const int r16 = lane & 15, q = lane >> 4;
    const int32_t K = a.k;
    const int nkb = K / BKB;
    auto swz = [](int r) __attribute__((always_inline)) { return (r / RPW) & (CPR - 1); };
    // fragment offsets of the wave's first block of 16 rows, k-step 0.  Step s reads logical chunk
    // 4s + q: xor (4s << 4) commutes with the swizzle; block i lies 16 rows further on, where the swizzle repeats.
    static_assert((16 / RPW) % CPR == 0, "the swizzle must repeat every 16 rows");
    constexpr int BLKP = 16 * BKB, BLKQ = 16 * BKB;        // (K-major operands; the others: tr_frag below)
    const int rp0 = wr * TR * 32 + r16, rq0 = wc * TC * 32 + r16;
    const int offP0 = rp0 * BKB + ((q ^ swz(rp0)) << 4);
    const int offQ0 = BR * BKB + rq0 * BKB + ((q ^ swz(rq0)) << 4);
    // without slabs on their way the waits below count only loads: let the previous tile's stores finish first
    if (!have_slabs) wait_vmcnt<0>();
    Dma dma(a, lds_base, cur_item, nxt_item, wave, lane, ring);
    const uint32_t b = cur_item.b;
    const int32_t j0 = cur_item.j0, i0 = cur_item.i0;
    const bool ahead = dma.ahead;
    const int nk = dma.nk, LD = dma.LD, ring0 = dma.ring0;
    auto dma1 = [&](auto dc, int kt, auto tailc, int stage) __attribute__((always_inline)) {
        dma.template issue<decltype(dc)::value, decltype(tailc)::value>(kt, stage);
    };

    // the dequantisation scales of this lane's outputs, fetched now so that the epilogue does
    // not wait on memory between its stores
    half_t sxh[AR];
    half4_t syh[AC];
    if (FUSED) {
#pragma unroll
        for (int i = 0; i < AR; ++i) {
            const int32_t row = min(j0 + wr * TR * 32 + i * 16 + r16, a.n - 1);
            sxh[i] = a.srow ? a.srow[a.bc_row ? row : (int64_t)b * a.n + row] : (half_t)1.0f;
        }
#pragma unroll
        for (int j = 0; j < AC; ++j) {
            const int32_t col = min(i0 + wc * TC * 32 + j * 16 + q * 4, a.m - 4);   // m % 4 == 0
            syh[j] = a.scol ? *reinterpret_cast<const half4_t*>(a.scol + (a.bc_col ? 0 : (int64_t)b * a.m) + col) : half4_t{1, 1, 1, 1};
        }
    }

    // kEpiSumI8: the scales of this wave's rows for every entry of the sum wait in its output strip, idle until the epilogue
    if constexpr (FOLD) {
        constexpr int WROWS = TR * 32;
        for (int t = lane; t < a.nsum * WROWS; t += 64) {
            const int32_t row = min(j0 + wr * WROWS + t % WROWS, a.n - 1);
            *reinterpret_cast<half_t*>(stg + t * 2) = a.srow[((int64_t)b * a.nsum + t / WROWS) * a.n + row];
        }
    }
    float4_t facc[FOLD ? AR : 1][FOLD ? AC : 1];
    if constexpr (FOLD) {
#pragma unroll
        for (int i = 0; i < AR; ++i)
#pragma unroll
            for (int j = 0; j < AC; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) facc[i][j][e] = 0.0f;
    }
    acc_t acc[AR][AC];
#pragma unroll
    for (int i = 0; i < AR; ++i)
#pragma unroll
        for (int j = 0; j < AC; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = 0;
    if constexpr ((LAY & 4) != 0 && !REST) {
        const int32_t K1 = nkb * BKB, rem = K - K1;
        for (int32_t eb = 0; eb < (SUM ? a.nsum : 1) && rem > 0; ++eb) {
            const int64_t be = SUM ? (int64_t)b * a.nsum + eb : (int64_t)b;
            const int8_t* Pr = a.P + be * a.strideP + K1;
            const int8_t* Qr = a.Q + be * a.strideQ + K1;
            // bytes [kc, kc + 16) of the rest of a row, zeros from byte `rem` on: the piece may start at any address and
            // end inside (rows of K that are whole dwords, not whole 16-byte pieces)
            struct __attribute__((packed, aligned(1))) Piece16 { uint32_t x, y, z, w; };
            // (without branches -- a load under a condition would be waited for before the next one is issued: the 16 bytes
            // that end where the piece or K ends, moved down by the dwords that lie beyond K)
            auto piece = [&](const int8_t* rest, int32_t kc) __attribute__((always_inline)) {
                if constexpr ((LAY & 8) == 0) {      // whole pieces only: one load under one condition
                    int4_t v = {0, 0, 0, 0};
                    if (kc < rem) {
                        const Piece16 t = *reinterpret_cast<const Piece16*>(rest + kc);
                        v = int4_t{(int32_t)t.x, (int32_t)t.y, (int32_t)t.z, (int32_t)t.w};
                    }
                    return v;
                }
                const int32_t over = min(max(kc + 16 - rem, 0), 16);        // bytes of the piece beyond K: 0, 4 ... 16
                const Piece16 t = *reinterpret_cast<const Piece16*>(rest + min(kc - over, rem - 16));       // (inside the row: at least one slab precedes `rest`)
                const int32_t w[8] = {(int32_t)t.x, (int32_t)t.y, (int32_t)t.z, (int32_t)t.w, 0, 0, 0, 0};
                const int sh = over >> 2;
                int4_t v;
#pragma unroll
                for (int d = 0; d < 4; ++d) v[d] = sh == 0 ? w[d] : sh == 1 ? w[d + 1] : sh == 2 ? w[d + 2] : sh == 3 ? w[d + 3] : 0;
                return v;
            };
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                if (ks * 64 < rem) {
                    const int32_t kc = ks * 64 + q * 16;
                    int4_t rp[AR], rq[AC];
#pragma unroll
                    for (int i = 0; i < AR; ++i) rp[i] = piece(Pr + (int64_t)min(j0 + wr * TR * 32 + i * 16 + r16, a.n - 1) * K, kc);
#pragma unroll
                    for (int j = 0; j < AC; ++j) rq[j] = piece(Qr + (int64_t)min(i0 + wc * TC * 32 + j * 16 + r16, a.m - 1) * K, kc);
#pragma unroll
                    for (int i = 0; i < AR; ++i)
#pragma unroll
                        for (int j = 0; j < AC; ++j) {
                            if constexpr (F16)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, rq[j]), __builtin_bit_cast(half8_t, rp[i]), acc[i][j], 0, 0, 0);
                            else
                                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(rq[j], rp[i], acc[i][j], 0, 0, 0);
                        }
                }
            }
        }
    }
    // Fragments: all AR of the row operand, and the column operand's in two sets of AC/2 -- a k-step is two
    // passes over the wave's rows, one per half of its columns, and while one set is multiplied the
    // other is read.  A row fragment's register is refilled with the next k-step's right after
    // its last MFMA of the second pass.
    constexpr int HC = AC / 2;
    int4_t fp[AR], fq[2][HC];
    // Transposing reads.  fp16 (ds_read_b64_tr_b16): within 16 lanes, lane j hands in the address of four halves -- row
    // of K k0 + j / 4, elements 4 (j % 4) .. + 3 of a block of 16 -- and lane i receives element i of rows k0 .. k0 + 3:
    // four consecutive values of K for its own row of the MFMA operand.  int8 (ds_read_b64_tr_b8): lane j hands in
    // eight bytes -- row of K k0 + j / 2, elements 8 (j % 2) .. + 7 -- and lane i receives element i of rows k0 .. k0 + 7.
    // Two reads per fragment either way, instead of eight 2-byte or sixteen 1-byte ones.  Block u (16 elements) of
    // row k lies at unit u ^ (k & 3) resp. u ^ (k & 7) (SlabDma, TSW): an exclusive-or of the block's offset with a
    // lane's constant.
    constexpr int ULOG = F16 ? 5 : 4;              // log2 of a block's bytes
    const int trx = F16 ? (r16 >> 2) << 5 : (r16 >> 1) << 4;                  // the exchange, as an offset
    const int trb = F16 ? (r16 & 3) << 3 : (r16 & 1) << 3;                    // the lane's eight bytes within the block
    const int trk = F16 ? q * 8 + (r16 >> 2) : q * 16 + (r16 >> 1);            // the row of K (within a k-step) this lane's first address names
    auto tr_frag = [&](const int8_t* part, int rowlen, int ublock, int ks) __attribute__((always_inline)) {
        // part: the operand's rows of K in the stage; rowlen: bytes per row of K; ublock: number of the block of 16 elements
        const uint32_t p0 = lds_base + (uint32_t)(part - smem) + (ks * (F16 ? 32 : 64) + trk) * rowlen + ((ublock << ULOG) ^ trx) + trb;
        const uint32_t p1 = p0 + (F16 ? 4 : 8) * rowlen;
        if constexpr (F16) {
            typedef short short4_t __attribute__((ext_vector_type(4)));
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p0);
            const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p1);
            return __builtin_bit_cast(int4_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
            typedef int int2_tv __attribute__((ext_vector_type(2)));
            const int2_tv lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) int2_tv*)(uintptr_t)p0);
            const int2_tv hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) int2_tv*)(uintptr_t)p1);
            return int4_t{lo.x, lo.y, hi.x, hi.y};
        }
    };
    auto lfragP = [&](auto ic, int stage, int ks) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (TRP) fp[i] = tr_frag(smem + stage * STAGE, BR * ESZ_IN, wr * TR * 2 + i, ks);
        else fp[i] = *reinterpret_cast<const int4_t*>(smem + stage * STAGE + (offP0 ^ (ks << 6)) + i * BLKP);
    };
    auto lfragQ = [&](auto setc, auto jjc, int stage, int ks) __attribute__((always_inline)) {       // fragment jj of column half `set`
        constexpr int set = decltype(setc)::value, jj = decltype(jjc)::value;
        constexpr int j = set * HC + jj;
        if constexpr (TRQ) fq[set][jj] = tr_frag(smem + stage * STAGE + BR * BKB, BC * ESZ_IN, wc * TC * 2 + j, ks);
        else fq[set][jj] = *reinterpret_cast<const int4_t*>(smem + stage * STAGE + (offQ0 ^ (ks << 6)) + j * BLKQ);
    };
    // One pass: the AR x HC MFMAs of column half `jh`, order pinned.  Between them the other set of column
    // fragments is read from k-step `qks` of stage `qs`; with REFILL the row fragments are refilled from
    // k-step `nks` of stage `ns`; and ND further memory operations (`memop`) are spread over the pass.
    // FIRST (kEpiSumI8): the pass starts the next entry's products; a tile's finished product goes into the sums right before its
    // accumulators start again from zero, eight vector operations under each MFMA of the wave beside it on the SIMD.
    constexpr int NMP = AR * HC;
    float fsx[FOLD ? AR : 1];            // FOLD: the scales of this lane's rows for the entry whose products are in the accumulators
    auto fold = [&](int i, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) facc[i][j][e] = __builtin_fmaf((float)acc[i][j][e], fsx[i], facc[i][j][e]);
        asm volatile("" : "+v"(facc[i][j]));
    };
    auto pass = [&](auto jhc, int qs, int qks, auto refillc, int ns, int nks, auto&& memop, auto nd_c, auto firstc) __attribute__((always_inline)) {
        constexpr int jh = decltype(jhc)::value, ND = decltype(nd_c)::value;
        constexpr bool REFILL = decltype(refillc)::value, FIRST = decltype(firstc)::value;
        static_for<0, NMP>([&](auto xc) __attribute__((always_inline)) {
            constexpr int x = decltype(xc)::value;
            constexpr int i = x / HC, jj = x % HC;
            if constexpr (FIRST) {
                fold(i, jh * HC + jj);
                acc[i][jh * HC + jj] = acc_t{0, 0, 0, 0};
            }
            // MFMA "A" = column-operand rows, "B" = row-operand rows: lane l, register e of the
            // result is output row l%16, column (l/16)*4 + e of the 16x16 tile
            if constexpr (F16)      // 64 bytes of K are 32 halves: same lane -> byte assignment as the int8 MFMA
                acc[i][jh * HC + jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, fq[jh][jj]),
                                                                              __builtin_bit_cast(half8_t, fp[i]), acc[i][jh * HC + jj], 0, 0, 0);
            else
                acc[i][jh * HC + jj] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fq[jh][jj], fp[i], acc[i][jh * HC + jj], 0, 0, 0);
            if constexpr (REFILL && jj == HC - 1) lfragP(std::integral_constant<int, i>{}, ns, nks);
            if constexpr (x % AR == 0 && x / AR < HC)
                lfragQ(std::integral_constant<int, 1 - jh>{}, std::integral_constant<int, x / AR>{}, qs, qks);
            constexpr int lo = (x * ND) / NMP, hi = ((x + 1) * ND) / NMP;
            static_for<lo, hi>([&](auto yc) __attribute__((always_inline)) { memop(yc); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    auto no_memop = [](auto) __attribute__((always_inline)) {};

    dma.prime(have_slabs);
    if (FUSED) {     // pin the scale loads above the K loop (the waits just above cover them)
#pragma unroll
        for (int i = 0; i < AR; ++i) asm volatile("" : "+v"(sxh[i]));
#pragma unroll
        for (int j = 0; j < AC; ++j) asm volatile("" : "+v"(syh[j]));
        // parked in this wave's output strip, idle until the epilogue: fewer registers live across the K loop
#pragma unroll
        for (int i = 0; i < AR; ++i) *reinterpret_cast<half_t*>(stg + (i * 64 + lane) * 2) = sxh[i];
#pragma unroll
        for (int j = 0; j < AC; ++j) *reinterpret_cast<half4_t*>(stg + 1024 + (j * 64 + lane) * 8) = syh[j];
    }
    static_for<0, AR>([&](auto xc) __attribute__((always_inline)) { lfragP(xc, ring0, 0); });
    static_for<0, HC>([&](auto xc) __attribute__((always_inline)) { lfragQ(I0{}, xc, ring0, 0); });

    int cur = ring0;
    // tail slab index: it + LD - nk of the next tile, or nk - 1 of this one
    const int tmul = ahead ? 1 : 0, tadd = ahead ? LD - nk : nk - 1;
    auto slab = [&](int it, auto tailc, auto firstc) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tailc)::value;
        const int nxt = cur + 1 == NST ? 0 : cur + 1;
        static_for<0, KS - 1>([&](auto ksc) __attribute__((always_inline)) {
            constexpr int ks = decltype(ksc)::value;
            constexpr std::integral_constant<bool, decltype(firstc)::value && ks == 0> start{};
            pass(I0{}, cur, ks, std::false_type{}, 0, 0, no_memop, I0{}, start);
            pass(I1{}, cur, ks + 1, std::true_type{}, cur, ks + 1, no_memop, I0{}, start);
        });
        pass(I0{}, cur, KS - 1, std::false_type{}, 0, 0, no_memop, I0{}, std::false_type{});       // the last reads of stage cur
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<(NST - 2) * CNT>();       // slab it + 1 has landed (with fewer slabs than stages it had before the loop)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        const int kt2 = TAIL ? (REST ? max(it * tmul + tadd, dma.first) : it * tmul + tadd) : it + LD;
        const int tgt = cur + LD >= NST ? cur + LD - NST : cur + LD;       // the stage slab it + LD belongs to
        pass(I1{}, nxt, 0, std::true_type{}, nxt, 0,
             [&](auto dc) __attribute__((always_inline)) { dma1(dc, kt2, tailc, tgt); },
             std::integral_constant<int, CNT>{}, std::false_type{});
        if constexpr (SUM) dma.advance();
        __builtin_amdgcn_sched_barrier(0);
        cur = nxt;
    };
    int it = 0;
    if constexpr (SUM) dma.seek(false, min(LD, nk - 1));
    if constexpr (FOLD) {
        // One loop for the slabs before the tail and the tail's (what they request follows Pk / Qk), two bodies: an entry's first slab
        // and its others.
        static_assert(KS > 1, "an entry starts in a k-step of its own");
        auto next_slab = [&](auto firstc) __attribute__((always_inline)) {
            if (it == nk - LD) {
                dma.retarget();
                dma.seek(true, ahead ? 0 : nk - 1);
            }
            slab(it, std::false_type{}, firstc);
            ++it;
        };
#pragma unroll
        for (int i = 0; i < AR; ++i) fsx[i] = 0.0f;
        for (int entry = 0; entry < a.nsum; ++entry) {
            next_slab(std::true_type{});
#pragma unroll
            for (int i = 0; i < AR; ++i) fsx[i] = (float)*reinterpret_cast<const half_t*>(stg + (entry * TR * 32 + i * 16 + r16) * 2);
            for (int s = 1; s < nkb; ++s) next_slab(std::false_type{});
        }
#pragma unroll
        for (int i = 0; i < AR; ++i)
#pragma unroll
            for (int j = 0; j < AC; ++j) fold(i, j);
    } else {
        auto plain = [&](int t, auto tailc) __attribute__((always_inline)) { slab(t, tailc, std::false_type{}); };
        for (; it < nk - LD; ++it) plain(it, std::false_type{});       // slabs LD .. nk-1 of this tile follow
        if constexpr (SUM) dma.seek(true, ahead ? 0 : nk - 1);
        tail_slabs<REST>(dma, it, plain);                              // then the tail's
    }
    if (!ahead) wait_vmcnt<0>();         // drain the clamped loads before the ring is reused
    ring = cur;                          // (ring0 + nk) % NST: where the next tile's slab 0 is, or will be put

    const int64_t obase = (int64_t)b * a.n * a.m;
    using Out = StripOut<EPI, TC, (LAY & 16) != 0>;       // the results leave through this wave's strip of LDS
    constexpr int NCH = Out::NCH, RB = Out::RB;
    auto slot = [](int r, int p) __attribute__((always_inline)) { return Out::slot(r, p); };
    half_t sxr[AR];
    half4_t syr[AC];
    if (FUSED) {      // the scales come back from the strip before the results overwrite it
#pragma unroll
        for (int i = 0; i < AR; ++i) sxr[i] = *reinterpret_cast<const half_t*>(stg + (i * 64 + lane) * 2);
#pragma unroll
        for (int j = 0; j < AC; ++j) syr[j] = *reinterpret_cast<const half4_t*>(stg + 1024 + (j * 64 + lane) * 8);
#pragma unroll
        for (int i = 0; i < AR; ++i) asm volatile("" : "+v"(sxr[i]));
#pragma unroll
        for (int j = 0; j < AC; ++j) asm volatile("" : "+v"(syr[j]));
    }
#pragma unroll
    for (int i = 0; i < TR; ++i) {        // blocks of 32 output rows: two rows of MFMA tiles
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int srow = h * 16 + r16;      // row of the strip
                if constexpr (epi_out32(EPI)) {
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj) {
                        int4_t v;
                        if constexpr (FOLD) v = __builtin_bit_cast(int4_t, facc[2 * i + h][2 * c + jj]);
                        else v = __builtin_bit_cast(int4_t, acc[2 * i + h][2 * c + jj]);
                        *reinterpret_cast<int4_t*>(stg + srow * RB + slot(srow, jj * 4 + q)) = v;
                    }
                } else {
                    float sx = 0.0f;
                    if (FUSED) sx = (float)sxr[2 * i + h];
#pragma unroll
                    for (int j = 0; j < AC; ++j) {
                        half4_t hv;
                        if constexpr (FOLD) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) hv[e] = (half_t)facc[2 * i + h][j][e];
                        } else if constexpr (F16) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) hv[e] = (half_t)acc[2 * i + h][j][e];
                        } else {
                            const half4_t sy = syr[j];
#pragma unroll
                            for (int e = 0; e < 4; ++e) hv[e] = dequant(acc[2 * i + h][j][e], sx, (float)sy[e]);
                        }
                        *reinterpret_cast<half4_t*>(stg + srow * RB + slot(srow, j * 2 + (q >> 1)) + (q & 1) * 8) = hv;
                    }
                }
            }
            Out::store_rows(a, stg, obase, j0 + wr * TR * 32 + i * 32, i0 + wc * TC * 32 + c * 32, lane);
        }
    }
    return ahead;
}

// The same tile with v_mfma_i32_32x32x32_i8 / v_mfma_f32_32x32x16_f16 (k-steps of 32 bytes, a wave owns
// TR x TC tiles of 32x32, lane l holds output row l%32; both operands' fragments double buffered,
// the barrier before the last k-step).  Used where a wave's share of a k-step is too small for the
// row fragments' refill-after-last-use above to hide the LDS latency (the 128x128 and smaller
// workgroup tiles, one wave per SIMD) and for products of a single slab.  DMA, ring and tail are
// the ones described above.
template <int WR, int WC, int TR, int TC, int BKB, int EPI, int NST, int LAY = 0>
__device__ __forceinline__ bool gemm_dma_tile32(const GemmArgs& a, int8_t* smem, int8_t* stg, uint32_t lds_base,
                                              const GemmItem cur_item, const GemmItem nxt_item, const bool have_slabs, int& ring) {
    constexpr bool FUSED = EPI == kEpiDequant, F16 = epi_f16(EPI);
    static_assert(!epi_sum(EPI), "sums over the batch: the 16x16 form");
    constexpr bool PT = (LAY & 1) != 0, QT = (LAY & 2) != 0;
    static_assert((LAY & 3) == 0 || BKB == 128, "transposed operands: 128 bytes of K per slab");
    constexpr int ESZ_IN = F16 ? 2 : 1;            // bytes per operand element
    using acc_t = std::conditional_t<F16, float16_tv, int16_tv>;
    constexpr int KS = BKB / 32, CPR = BKB / 16;
    constexpr int NW = WR * WC, BR = WR * TR * 32, BC = WC * TC * 32;
    constexpr bool TRP = PT, TRQ = QT;             // fragments of a (K, L) operand: transposing LDS reads
    // The rest of a depth that is not whole slabs is a slab of its own: beside an operand stored (K, rows), whose fragments would
    // have to be gathered two bytes at a time (64 x 500 x 500 over 1024 heads: 161 -> 132 us, 500 x 80 x 500 289 -> 243 us), and in the
    // small tiles (500 x 500 x 64 over 512 heads 105 -> 93 us).  256 x 256 tiles of K-major operands are bound by their products and
    // multiply no slab that is mostly zeros: 16 x 1000^3 60.4 us, 62.1 us so.
    constexpr bool REST = (LAY & 4) != 0 && (PT || QT || BR * BC < 256 * 256);
    using Dma = SlabDma<BR, BC, BKB, NW, NST, LAY, F16, TRP || TRQ, false, REST>;
    constexpr int STAGE = Dma::STAGE, CNT = Dma::CNT;      // bytes per ring stage; DMA instructions per wave and slab
    constexpr int NM = TR * TC;
    constexpr int RPW = 256 / BKB;                 // rows per 256-byte bank wrap
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC;
    const int lrow = lane & 31, lk = lane >> 5;
    const int32_t K = a.k;
    auto swz = [](int r) __attribute__((always_inline)) { return (r / RPW) & (CPR - 1); };
    // fragment offsets for k-step 0; step s reads logical chunk 2s + lk: xor (2s << 4) commutes with the swizzle
    int offP[TR], offQ[TC];
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        const int r = wr * TR * 32 + i * 32 + lrow;
        offP[i] = r * BKB + ((lk ^ swz(r)) << 4);          // (K-major operands; the others: tr_frag below)
    }
#pragma unroll
    for (int j = 0; j < TC; ++j) {
        const int r = wc * TC * 32 + j * 32 + lrow;
        offQ[j] = BR * BKB + r * BKB + ((lk ^ swz(r)) << 4);
    }
    // without slabs on their way the waits below count only loads: let the previous tile's stores finish first
    if (!have_slabs) wait_vmcnt<0>();
    Dma dma(a, lds_base, cur_item, nxt_item, wave, lane, ring);
    const uint32_t b = cur_item.b;
    const int32_t j0 = cur_item.j0, i0 = cur_item.i0;
    const bool ahead = dma.ahead;
    const int nk = dma.nk, LD = dma.LD, ring0 = dma.ring0;
    auto dma1 = [&](auto dc, int kt, auto tailc, int stage) __attribute__((always_inline)) {
        dma.template issue<decltype(dc)::value, decltype(tailc)::value>(kt, stage);
    };

    // the dequantisation scales of this lane's outputs, fetched now so that the epilogue does
    // not wait on memory between its stores
    half_t sxh[TR];
    half4_t syh[TC][4];
    if (FUSED) {
#pragma unroll
        for (int i = 0; i < TR; ++i) {
            const int32_t row = min(j0 + wr * TR * 32 + i * 32 + lrow, a.n - 1);
            sxh[i] = a.srow ? a.srow[a.bc_row ? row : (int64_t)b * a.n + row] : (half_t)1.0f;
        }
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int32_t col = min(i0 + wc * TC * 32 + j * 32 + g4 * 8 + lk * 4, a.m - 4);   // m % 4 == 0
                syh[j][g4] = a.scol ? *reinterpret_cast<const half4_t*>(a.scol + (a.bc_col ? 0 : (int64_t)b * a.m) + col) : half4_t{1, 1, 1, 1};
            }
    }

    acc_t acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
    if constexpr ((LAY & 4) != 0 && !REST) {
        // The depth beyond the last whole slab, as in the 16x16 form.  Pieces may start at any address and end inside (rows of K
        // that are whole dwords, not whole 16-byte pieces).
        const int32_t K1 = nk * BKB, rem = K - K1;           // bytes
        if (rem > 0) {
            struct __attribute__((packed, aligned(1))) Piece16 { uint32_t x, y, z, w; };
            const int8_t* Pr = a.P + (int64_t)b * a.strideP;
            const int8_t* Qr = a.Q + (int64_t)b * a.strideQ;
            // a K-major operand's piece: bytes [kc, kc + 16) of the rest of row `row`, zeros from byte `rem` on
            // (without branches -- a load under a condition would be waited for before the next one is issued.  The
            // piece: the 16 bytes that end where the piece or K ends, moved down by the dwords that lie beyond K.)
            auto piece = [&](const int8_t* base, int32_t row, int32_t kc) __attribute__((always_inline)) {
                if constexpr ((LAY & 8) == 0) {      // whole pieces only: one load under one condition (15 % quicker than the form below where it applies)
                    int4_t v = {0, 0, 0, 0};
                    if (kc < rem) {
                        const Piece16 t = *reinterpret_cast<const Piece16*>(base + (int64_t)row * K + K1 + kc);
                        v = int4_t{(int32_t)t.x, (int32_t)t.y, (int32_t)t.z, (int32_t)t.w};
                    }
                    return v;
                }
                const int32_t over = min(max(kc + 16 - rem, 0), 16);        // bytes of the piece beyond K: 0, 4 ... 16
                const Piece16 t = *reinterpret_cast<const Piece16*>(base + (int64_t)row * K + K1 + min(kc - over, rem - 16));      // (inside the row: at least one slab precedes)
                const int32_t w[8] = {(int32_t)t.x, (int32_t)t.y, (int32_t)t.z, (int32_t)t.w, 0, 0, 0, 0};
                const int sh = over >> 2;
                int4_t v;
#pragma unroll
                for (int d = 0; d < 4; ++d) v[d] = sh == 0 ? w[d] : sh == 1 ? w[d + 1] : sh == 2 ? w[d + 2] : sh == 3 ? w[d + 3] : 0;
                return v;
            };
            auto load_ks = [&](int4_t (&rp)[TR], int4_t (&rq)[TC], int ks) __attribute__((always_inline)) {
                const int32_t kc = ks * 32 + lk * 16;
#pragma unroll
                for (int i = 0; i < TR; ++i) {
                    const int32_t row = min(j0 + wr * TR * 32 + i * 32 + lrow, a.n - 1);
                    rp[i] = int4_t{0, 0, 0, 0};
                    if (ks * 32 < rem) rp[i] = piece(Pr, row, kc);
                }
#pragma unroll
                for (int j = 0; j < TC; ++j) {
                    const int32_t col = min(i0 + wc * TC * 32 + j * 32 + lrow, a.m - 1);
                    rq[j] = int4_t{0, 0, 0, 0};
                    if (ks * 32 < rem) rq[j] = piece(Qr, col, kc);
                }
            };
            auto mac_ks = [&](const int4_t (&rp)[TR], const int4_t (&rq)[TC], int ks) __attribute__((always_inline)) {
                if (ks * 32 < rem) {
#pragma unroll
                    for (int i = 0; i < TR; ++i)
#pragma unroll
                        for (int j = 0; j < TC; ++j) {
                            if constexpr (F16)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, rq[j]), __builtin_bit_cast(half8_t, rp[i]), acc[i][j], 0, 0, 0);
                            else
                                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(rq[j], rp[i], acc[i][j], 0, 0, 0);
                        }
                }
            };
            // a k-step at a time, which keeps the wide accumulator tiles of this form in registers
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                int4_t rp[TR], rq[TC];
                load_ks(rp, rq, ks);
                mac_ks(rp, rq, ks);
            }
        }
    }
    int4_t fp[2][TR], fq[2][TC];
    // Transposing reads as in the 16x16 form.  Here a fragment is 32 rows x 16 bytes of K: the wave's four groups of
    // 16 lanes are (rows 0-15 | 16-31) x (first | second half of the k-step's 32 bytes), so a group's block of 16
    // rows is number 2 i + (group & 1) of the wave's, and its rows of K start at 8 (fp16) or 16 (int8) times group >> 1.
    constexpr int ULOG = F16 ? 5 : 4;              // log2 of a block's bytes
    const int trj = lane & 15, trg = lane >> 4;
    const int trx = F16 ? (trj >> 2) << 5 : (trj >> 1) << 4;                  // the exchange, as an offset
    const int trb = F16 ? (trj & 3) << 3 : (trj & 1) << 3;                    // the lane's eight bytes within the block
    const int trk = F16 ? (trg >> 1) * 8 + (trj >> 2) : (trg >> 1) * 16 + (trj >> 1);      // the row of K (within a k-step) of the lane's first address
    auto tr_frag = [&](const int8_t* part, int rowlen, int ublock0, auto ic, int ks) __attribute__((always_inline)) {
        // part: the operand's rows of K in the stage; rowlen: bytes per row of K; ublock0: number of the wave's first block of 16 elements
        constexpr int i = decltype(ic)::value;
        const uint32_t p0 = lds_base + (uint32_t)(part - smem) + (ks * (F16 ? 16 : 32) + trk) * rowlen + (((ublock0 + 2 * i + (trg & 1)) << ULOG) ^ trx) + trb;
        const uint32_t p1 = p0 + (F16 ? 4 : 8) * rowlen;
        if constexpr (F16) {
            typedef short short4_t __attribute__((ext_vector_type(4)));
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p0);
            const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p1);
            return __builtin_bit_cast(int4_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
            typedef int int2_tv __attribute__((ext_vector_type(2)));
            const int2_tv lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) int2_tv*)(uintptr_t)p0);
            const int2_tv hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) int2_tv*)(uintptr_t)p1);
            return int4_t{lo.x, lo.y, hi.x, hi.y};
        }
    };
    auto lfrag1 = [&](auto xc, auto bufc, int stage, int ks) __attribute__((always_inline)) {
        constexpr int x = decltype(xc)::value, buf = decltype(bufc)::value;
        if constexpr (x < TR) {
            if constexpr (TRP) {
                fp[buf][x] = tr_frag(smem + stage * STAGE, BR * ESZ_IN, wr * TR * 2, std::integral_constant<int, x>{}, ks);
            } else {
                fp[buf][x] = *reinterpret_cast<const int4_t*>(smem + stage * STAGE + (offP[x] ^ (ks << 5)));
            }
        } else {
            if constexpr (TRQ) {
                fq[buf][x - TR] = tr_frag(smem + stage * STAGE + BR * BKB, BC * ESZ_IN, wc * TC * 2, std::integral_constant<int, x - TR>{}, ks);
            } else {
                fq[buf][x - TR] = *reinterpret_cast<const int4_t*>(smem + stage * STAGE + (offQ[x - TR] ^ (ks << 5)));
            }
        }
    };
    // one k-step: NM MFMAs with NMEM memory operations spread evenly between them, order pinned
    auto kstep = [&](auto bufc, auto&& memop, auto nmem_c) __attribute__((always_inline)) {
        constexpr int NMEM = decltype(nmem_c)::value, buf = decltype(bufc)::value;
        static_for<0, NM>([&](auto xc) __attribute__((always_inline)) {
            constexpr int x = decltype(xc)::value;
            constexpr int i = x / TC, j = x % TC;
            // MFMA "A" = column-operand rows, "B" = row-operand rows: lane l, register e of the
            // result is output row l%32, column (e/4)*8 + (l/32)*4 + e%4 of the 32x32 tile
            if constexpr (F16)      // 32 bytes of K are 16 halves: same lane -> byte assignment as the int8 MFMA
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, fq[buf][j]),
                                                                   __builtin_bit_cast(half8_t, fp[buf][i]), acc[i][j], 0, 0, 0);
            else
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fq[buf][j], fp[buf][i], acc[i][j], 0, 0, 0);
            constexpr int lo = (x * NMEM) / NM, hi = ((x + 1) * NMEM) / NM;
            static_for<lo, hi>([&](auto yc) __attribute__((always_inline)) { memop(yc); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using C0 = std::integral_constant<int, 0>;

    dma.prime(have_slabs);
    if (FUSED) {     // pin the scale loads above the K loop (the waits just above cover them)
#pragma unroll
        for (int i = 0; i < TR; ++i) asm volatile("" : "+v"(sxh[i]));
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) asm volatile("" : "+v"(syh[j][g4]));
        // parked in this wave's output strip, idle until the epilogue: 20 fewer registers live across the K loop
#pragma unroll
        for (int i = 0; i < TR; ++i) *reinterpret_cast<half_t*>(stg + (i * 64 + lane) * 2) = sxh[i];
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) *reinterpret_cast<half4_t*>(stg + 1024 + lk * 64 + (j * 4 + g4) * 8) = syh[j][g4];
    }
    static_for<0, TR + TC>([&](auto xc) __attribute__((always_inline)) { lfrag1(xc, C0{}, ring0, 0); });

    int cur = ring0;
    // tail slab index: it + LD - nk of the next tile, or nk - 1 of this one
    const int tmul = ahead ? 1 : 0, tadd = ahead ? LD - nk : nk - 1;
    auto slab = [&](int it, auto tailc) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tailc)::value;
        const int nxt = cur + 1 == NST ? 0 : cur + 1;
        static_for<0, KS - 1>([&](auto ksc) __attribute__((always_inline)) {
            constexpr int ks = decltype(ksc)::value;
            kstep(std::integral_constant<int, (ks & 1)>{},
                  [&](auto xc) __attribute__((always_inline)) {
                      lfrag1(xc, std::integral_constant<int, ((ks + 1) & 1)>{}, cur, ks + 1);
                  },
                  std::integral_constant<int, TR + TC>{});
        });
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<(NST - 2) * CNT>();       // slab it + 1 has landed (with fewer slabs than stages it had before the loop)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        const int kt2 = TAIL ? (REST ? max(it * tmul + tadd, dma.first) : it * tmul + tadd) : it + LD;
        const int tgt = cur + LD >= NST ? cur + LD - NST : cur + LD;       // the stage slab it + LD belongs to
        kstep(std::integral_constant<int, ((KS - 1) & 1)>{},
              [&](auto xc) __attribute__((always_inline)) {
                  constexpr int x = decltype(xc)::value;
                  if constexpr (x < TR + TC) lfrag1(xc, std::integral_constant<int, (KS & 1)>{}, nxt, 0);
                  else dma1(std::integral_constant<int, x - (TR + TC)>{}, kt2, tailc, tgt);
              },
              std::integral_constant<int, TR + TC + CNT>{});
        __builtin_amdgcn_sched_barrier(0);
        cur = nxt;
    };
    int it = 0;
    for (; it < nk - LD; ++it) slab(it, std::false_type{});       // slabs LD .. nk-1 of this tile follow
    tail_slabs<REST>(dma, it, slab);                              // then the tail's
    if (!ahead) wait_vmcnt<0>();         // drain the clamped loads before the ring is reused
    ring = cur;                          // (ring0 + nk) % NST: where the next tile's slab 0 is, or will be put

    const int64_t obase = (int64_t)b * a.n * a.m;
    using Out = StripOut<EPI, TC, (LAY & 16) != 0>;       // the results leave through this wave's strip of LDS
    constexpr int NCH = Out::NCH, RB = Out::RB;
    auto slot = [](int r, int p) __attribute__((always_inline)) { return Out::slot(r, p); };
    half_t sxr[TR];
    half4_t syr[TC][4];
    if (FUSED) {      // the scales come back from the strip before the results overwrite it
#pragma unroll
        for (int i = 0; i < TR; ++i) sxr[i] = *reinterpret_cast<const half_t*>(stg + (i * 64 + lane) * 2);
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) syr[j][g4] = *reinterpret_cast<const half4_t*>(stg + 1024 + lk * 64 + (j * 4 + g4) * 8);
#pragma unroll
        for (int i = 0; i < TR; ++i) asm volatile("" : "+v"(sxr[i]));
#pragma unroll
        for (int j = 0; j < TC; ++j)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) asm volatile("" : "+v"(syr[j][g4]));
    }
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        float sx = 0.0f;
        if (FUSED) sx = (float)sxr[i];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            if constexpr (epi_out32(EPI)) {
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    int4_t v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const auto x = acc[i][c][g4 * 4 + e];       // (a value of its own: the cast of a vector's element takes the first one)
                        v[e] = __builtin_bit_cast(int32_t, x);
                    }
                    *reinterpret_cast<int4_t*>(stg + lrow * RB + slot(lrow, g4 * 2 + lk)) = v;
                }
            } else {
#pragma unroll
                for (int j = 0; j < TC; ++j)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        half4_t h;
                        if constexpr (F16) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[i][j][g4 * 4 + e];
                        } else {
                            const half4_t sy = syr[j][g4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) h[e] = dequant(acc[i][j][g4 * 4 + e], sx, (float)sy[e]);
                        }
                        *reinterpret_cast<half4_t*>(stg + lrow * RB + slot(lrow, j * 4 + g4) + lk * 8) = h;
                    }
            }
            Out::store_rows(a, stg, obase, j0 + wr * TR * 32 + i * 32, i0 + wc * TC * 32 + c * 32, lane);
        }
    }
    return ahead;
}

// Persistent kernel: WR x WC waves, wave tile = TR x TC blocks of 32x32 outputs, computed with the
// 16x16 MFMAs (MF = 16) or the 32x32 ones (MF = 32).  Workgroup w of G
// takes items round*G + (w%8)*(G/8) + w/8: the workgroups of one XCD (w % 8) work on adjacent
// tiles and share operand slabs in that XCD's L2.  When the tile count leaves a last round
// that at most half the workgroups could join, those tiles are issued as row halves (HALVES), one
// per workgroup: a wave then owns TR/2 x TC blocks, which keeps the fragment reads per MFMA
// lower than halving the columns would.
// (the sums over the batch hold two sets of accumulators: two waves a SIMD, so that the folding of one passes under the
// products of the other)
template <int WR, int WC, int TR, int TC, int BKB, int EPI, bool HALVES, int NST, int LAY, int MF>
__global__ __launch_bounds__(WR* WC * 64, epi_fold(EPI) ? 2 : 1) void k_gemm_dma(DmaArgs da) {
    static_assert(!(HALVES && (LAY & 4) != 0), "half tiles only where the depth is whole slabs");
    static_assert(MF == 16 || MF == 32, "MFMA tile");
    constexpr int BR = WR * TR * 32, BC = WC * TC * 32;
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t*)smem;
    // behind the operand ring: one 4 KB strip per wave for the output rows on their way out
    constexpr int STRIP = TC * 64 * 32 > 4096 ? TC * 64 * 32 : 4096;      // 32 rows of the widest chunk (fp16: TC*64 bytes, int32: 128)
    int8_t* stg = smem + NST * (BR + BC) * BKB + (threadIdx.x >> 6) * STRIP;
    const uint32_t G = gridDim.x;
    const uint32_t w = (G % 8 == 0) ? (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8 : blockIdx.x;
    bool have_slabs = false;
    int ring = 0;
    GemmItem cur = gemm_item<BR, BC>(w, da);
    for (uint32_t L = w; cur.valid; L += G) {
        const GemmItem nxt = gemm_item<BR, BC>(L + G, da);
        if (HALVES && cur.half) {
            if constexpr (HALVES) {
                if constexpr (MF == 16) have_slabs = gemm_dma_tile<WR, WC, TR / 2, TC, BKB, EPI, NST, LAY>(da.g, smem, stg, lds_base, cur, nxt, have_slabs, ring);
                else have_slabs = gemm_dma_tile32<WR, WC, TR / 2, TC, BKB, EPI, NST, LAY>(da.g, smem, stg, lds_base, cur, nxt, have_slabs, ring);
            }
        } else {
            if constexpr (MF == 16) have_slabs = gemm_dma_tile<WR, WC, TR, TC, BKB, EPI, NST, LAY>(da.g, smem, stg, lds_base, cur, nxt, have_slabs, ring);
            else have_slabs = gemm_dma_tile32<WR, WC, TR, TC, BKB, EPI, NST, LAY>(da.g, smem, stg, lds_base, cur, nxt, have_slabs, ring);
        }
        cur = nxt;
    }
}

// Ring stages: four for the 128x128 and 128x64 tile kernels, which finish a slab before a load from L2 returns (two, three,
// six and eight stages, and slabs of 64 or 256 bytes, all measured 1-3 us slower at 512 x 4096 x 4096); two for the
// 256x256 tile, whose ring then fills the LDS beside the output strips.
constexpr int kRingSmall = 4, kRingBig = 2;

template <int WR, int WC, int TR, int TC, int BKB, int EPI, bool HALVES, int NST, int LAY, int MF>
static int launch_dma_kernel(const DmaArgs& da, unsigned grid, hipStream_t st) {
    constexpr int BR = WR * TR * 32, BC = WC * TC * 32;
    constexpr int STRIP = TC * 64 * 32 > 4096 ? TC * 64 * 32 : 4096;
    constexpr int smem = NST * (BR + BC) * BKB + WR * WC * STRIP;      // operand ring + output strips
    static_assert(smem <= 160 * 1024, "LDS of one compute unit");
    auto kern = k_gemm_dma<WR, WC, TR, TC, BKB, EPI, HALVES, NST, LAY, MF>;
    static std::atomic<bool> lds_enabled[64];
    if (int e = enable_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_enabled)) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(WR * WC * 64), smem, st, da);
    return launch_status();
}

// MF: 16 = the 16x16 MFMAs (the large tile on products of several slabs), 32 = the 32x32 ones
// per_cu: workgroups a compute unit holds at once (their LDS and registers must allow it)
template <int WR, int WC, int TR, int TC, int BKB, int EPI, int NST, int LAY, int MF>
static int launch_dma(GemmArgs& a, int batch, hipStream_t st, int per_cu = 1) {
    constexpr int BR = WR * TR * 32, BC = WC * TC * 32;
    a.tiles_r = (int32_t)ceil_div(a.n, BR);
    a.tiles_c = (int32_t)ceil_div(a.m, BC);
    DmaArgs da;
    da.g = a;
    da.batch = batch;
    da.ntiles = a.tiles_r * a.tiles_c;
    const int64_t total = (int64_t)da.ntiles * batch;
    const int cus = compute_units() * per_cu;
    const int64_t grid = total < cus ? total : cus;
    // a last round of r <= grid/2 tiles is issued as 2r half tiles
    const int64_t r = total % grid;
    da.nfull = (uint32_t)total;
    da.nhalf = 0;
    // (a half tile's slab must split evenly over the waves too, and beside operands stored (K, rows) rows of K be whole 128-byte groups
    // in half a tile; a tile moved inside the matrix has no half of its own)
    constexpr bool F16 = epi_f16(EPI);
    if constexpr (TR % 2 == 0 && (LAY & (4 | 32)) == 0 && ((BR / 2 + BC) / (1024 / BKB)) % (WR * WC) == 0 &&
                  ((LAY & 3) == 0 || (BR / 2) * (F16 ? 2 : 1) % 128 == 0)) {
        if (r > 0 && 2 * r <= grid && (a.edge_in & 1) == 0) {
            da.nfull = (uint32_t)(total - r);
            da.nhalf = (uint32_t)(2 * r);
            return launch_dma_kernel<WR, WC, TR, TC, BKB, EPI, true, NST, LAY, MF>(da, (unsigned)grid, st);
        }
    }
    return launch_dma_kernel<WR, WC, TR, TC, BKB, EPI, false, NST, LAY, MF>(da, (unsigned)grid, st);
}

// A row operand stored (batch, n, k) beside a column operand that the batch shares: its entries, and the outputs', lie one behind the other
// and are one product of batch x n rows, whose tiles reach across the entries.  Entry by entry the last row tile of each is filled up to
// 128 rows, and the shared operand read for every entry: fp16, 16 entries of 32 x 8192 beside 4096 rows 127 -> 59 us, 7 of 300 x 1540 beside
// 7000 123 -> 67, the gradient of the 300 x 1540 117 -> 67; int8, 4 of 436 x 3712 beside 2304 29 -> 24.  (Operands stay below 4 GiB, what the tile kernels
// address; where it pays, join_gain.)
static bool rows_join(int batch, int32_t n, int64_t row_bytes) {
    return batch > 1 && (int64_t)batch * n < (1ll << 31) && batch * n * row_bytes < (1ll << 32);
}

// The same for a column operand stored (batch, m, k) beside a row operand that the batch shares: one product of batch x m columns, whose
// results go out to one matrix an entry (StripOut's SEG): 3 entries of 40 columns, 3904 x 12096, 34 -> 34 us and 12096 x 3904 28 -> 20; 5 of 136, the
// training step of a 3200 x 6848 ffn block 415 -> 369.
static bool cols_join(int batch, int32_t m, int64_t row_bytes) {
    return batch > 1 && (int64_t)batch * m < (1ll << 31) && batch * m * row_bytes < (1ll << 32) && (int64_t)batch * m * m < (1ll << 32);
}

// Tiles of 256 x 256, or those of the entries before they were joined (`apart`) where the joined product has more than two smaller ones a
// compute unit: fewer and fuller tiles are no reason to take those (16 entries of 960 columns, 640 x 2304, 192 large tiles apart, 180 joined
// or 600 small ones: 39, 37 and 45 us).
static int64_t big_tiles(int32_t n, int32_t m, int batch, int64_t apart, int64_t cus = compute_units()) {
    const int64_t big = ceil_div(n, 256) * ceil_div(m, 256) * batch;
    return apart > big && ceil_div(n, 128) * ceil_div(m, 128) * batch > 2 * cus ? apart : big;
}

// The time of a product's tiles, in tenths of a round of 128 x 128 tiles over the chip: a second round beside the first costs 0.8 of it (two
// workgroups fit a compute unit), a round of 256 x 256 tiles 2.2.  int8, K-major: `halves`, whether there are tiles of 128 x 64, a round of which is 0.8,
// and `whole`, whether a last round of large tiles is one of half tiles (fp16 products are drawn without: no better for it).
static int64_t tile_rounds(int32_t n, int32_t m, int batch, int64_t apart, bool whole, bool halves, int64_t cus) {
    const int64_t tiles = ceil_div(n, 128) * ceil_div(m, 128) * batch;
    if (n > 128 && m > 128 && big_tiles(n, m, batch, apart, cus) * 4 >= cus * 3) {
        const int64_t big = ceil_div(n, 256) * ceil_div(m, 256) * batch, r = big % cus;
        return whole && big > cus && r != 0 && 2 * r <= cus ? 22 * (big / cus) + 13 : 22 * ceil_div(big, cus);
    }
    if (halves && tiles * 4 < cus * 3 && ceil_div(n, 128) * ceil_div(m, 64) * batch <= cus) return 8;
    return tiles <= cus ? 10 : tiles <= 2 * cus ? 18 : 10 * ceil_div(tiles, cus);
}

// What joining entries does: rounds (tile_rounds) and 128 x 128 tiles, apart and joined.  Where it saves neither, the product apart is as quick or
// quicker: its results need no search for their entry (0.4 us on the smallest tiles), and fp16's few rows keep the kernels made for them.
// Over 1370 drawn int8 and 1430 fp16 products, joined : apart as a geometric mean,
//                   always                   where it saves rounds            (the better of both for each)
//   int8 rows       0.958, 102 worse > 4 %   0.949, 2 worse                   0.945
//   int8 columns    0.977, 273 worse         0.960, 4 worse                   0.958
//   fp16 rows       1.043, 307 worse         0.976, 6 worse                   0.961
//   fp16 columns    1.026, 335 worse         0.960, 3 worse                   0.958
// Where the rounds stay and tiles are saved it pays too at enough depth of whole slabs (fp16 rows: any from 1024 on); the same figures over those that the rules below take:
//   int8 rows 0.980, none of 103; fp16 rows 0.973, 2 of 120; int8 columns 0.964, 1 of 135; fp16 columns 0.948, none of 68, beside rows stored (K, rows) 0.944,
//   none of 26; rows from 1024 on where the tiles stay too 0.985, none of 19 (47 entries of 128 x 1280 beside 832 26.2 -> 22.8 us)
struct JoinGain {
    int64_t rounds, rounds_joined, tiles, tiles_joined, cus;
    bool fewer() const { return rounds_joined < rounds; }
    bool even(int64_t num, int64_t den) const { return rounds_joined == rounds && tiles_joined < tiles && tiles_joined * den <= tiles * num; }      // .. at most num / den of the tiles
};
static JoinGain join_gain(int32_t n, int32_t m, int batch, bool rows, int64_t apart, bool whole, bool halves) {
    const int32_t nj = rows ? n * batch : n, mj = rows ? m : m * batch;
    const int64_t cus = compute_units();       // (asked once: it is a call into the runtime)
    return {tile_rounds(n, m, batch, 0, whole, halves, cus), tile_rounds(nj, mj, 1, apart, whole, halves, cus), ceil_div(n, 128) * ceil_div(m, 128) * batch, ceil_div(nj, 128) * ceil_div(mj, 128), cus};
}
// fp16, whose few rows and short depths have kernels of their own: rows, past 128 of them or a depth of 448, or many tiles of enough depth
// (500 entries of 4 x 400 beside 314: 19.3 -> 7.5 us; 41 of 4 x 64 beside 3808, 4.3 apart and 5.7 joined)
static bool rows_join_pays_f16(int32_t n, int32_t m, int32_t k, bool kmajor, int batch, int64_t apart) {
    const JoinGain g = join_gain(n, m, batch, true, apart, false, false);
    if (k >= 1024 ? g.rounds_joined == g.rounds : kmajor && k % 64 == 0 && k >= 512 && g.even(1, 1)) return true;
    return g.fewer() && (n > 128 || k > 448 || (g.tiles > 4 * g.cus && g.tiles * k > 100000 && g.tiles_joined * 3 <= g.tiles));
}
// Columns, past 64 rows or a depth of 320; a row operand stored (K, rows) leaves fewer such calls to those kernels, and in a single round its long
// depths gain too (357 entries of 64 columns, 40 rows, K = 240 14.5 -> 9.5 us; 94 of 128, 64 rows, K = 2328 28.7 -> 23.7)
static bool cols_join_pays_f16(int32_t n, int32_t m, int32_t k, bool krows, int batch, int64_t apart) {
    const JoinGain g = join_gain(n, m, batch, false, apart, false, false);
    if (g.fewer() && (n > 64 || k > 320 || (krows && g.tiles * k > 19000 && g.tiles_joined * 4 <= g.tiles * 3))) return true;
    if (k % 64 == 0 && g.rounds >= 22 && (krows ? k >= 1024 && g.even(19, 20) : k >= 1536 && g.even(1, 1))) return true;
    return krows && n <= 64 && k >= 512 && g.tiles_joined <= g.cus;
}
// int8: rows also wherever the rounds stay, past one of them, with what the tiles of whole slabs do not take (19 of 2564 x 1600 beside 40 stored
// (K, columns), 495 -> 300; 37 of 128 x 36 beside 1280, 46 -> 17)
static bool rows_join_pays_i8(int32_t n, int32_t m, int32_t k, bool kmajor, int batch, int64_t apart) {
    const JoinGain g = join_gain(n, m, batch, true, apart, k % 64 == 0, kmajor && k % 128 == 0);
    if (kmajor && k % 128 == 0 && (k >= 1024 ? g.rounds_joined == g.rounds : k >= 384 && g.even(1, 1))) return true;
    return g.fewer() || ((!kmajor || k % 64 != 0) && g.tiles > g.cus && g.rounds_joined == g.rounds);
}
static bool cols_join_pays_i8(int32_t n, int32_t m, int32_t k, bool kmajor, int batch, int64_t apart) {
    const JoinGain g = join_gain(n, m, batch, false, apart, k % 64 == 0, kmajor && k % 128 == 0);
    if (kmajor && k % 128 == 0 && k >= 1536 && g.rounds >= 18 && (g.rounds > 18 || n >= 2048 ? g.even(19, 20) : g.even(17, 20))) return true;
    return g.fewer();
}

// gemm_parts.hip: parts that the depth of a product is divided into, 1 if it runs whole, else the time by its estimate in us as well; and that of one fp16 product of
// two operands stored (K, rows)
int32_t depth_parts(bool f16, int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, float* time = nullptr);
float krows_time(int32_t m, int32_t k, int32_t n);

}  // namespace cpmk
