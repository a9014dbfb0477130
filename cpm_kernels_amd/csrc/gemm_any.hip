// fp16 products of any size, layout and alignment: out[b, j, i] = sum_k P[b, j, k] Q[b, k, i], fp32 sums (cpm_kernels/torch/gemm.py:189-203).
// Each operand stored with K along its rows ("K-major": P (n, k), Q (m, k)) or with K as the row index (P (k, n), Q (k, m)).
//
// A workgroup is one tile of TR x TC outputs; it brings the next 64 of K into registers while the slab in LDS is multiplied.  A
// piece of eight inside its row moves whole at whatever address it lies (global accesses need no alignment), the one across a row's end
// in at most three narrower accesses, so that nothing asks for whole pieces.  Several workgroups a compute unit pass their
// waits under each other's work: bound by memory where there are enough of them and by a slab's latency elsewhere (1.1 us).
// Heads of 64 over 100 positions, 1024 of them: scores 20.8 -> 15.1 us, probabilities x values 20.8 -> 10.9, gradients of the values 19 -> 10.7 (3.6 to 5 TB/s;
// before: a kernel of 64 x 64 tiles that moved two to four elements at a time); 528 of 80 over 154: 48.5 -> 18.  gemm_f16_dispatch
// has where it is the better one beside the kernels with whole pieces.
#include "common.h"
#include <type_traits>

namespace cpmk {

struct AnyArgs {
    const half_t *P, *Q;           // a stride of 0 for one entry shared by the batch
    void* out;                     // (batch, n, m), fp16 or fp32
    int64_t strideP, strideQ;      // elements
    int32_t n, m, k;
    uint32_t tiles_r, tiles_c, tiles, first;      // tiles of a launch, number of its first one
};

// One operand's part of a slab: ROWS rows of the tile x 64 of K, in pieces of eight.
// K-major: LDS rows of 128 bytes, piece c of row r at c ^ (r & 7), read 16 bytes at a time.
// T (stored (K, rows)): LDS rows of ROWS halves, one for each of K; transposing reads (ds_read_b64_tr_b16): within 16 lanes, lane j hands in the
// address of four halves -- row of K k0 + j / 4, elements 4 (j % 4) .. + 3 of a block of 16 -- and lane i receives element i of rows
// k0 .. k0 + 3; block u (32 bytes) of row k lies at u ^ (k & 3).
template <bool T, int ROWS>
struct AnySlab {
    static constexpr int NP = ROWS * 64 / 8 / 256;                // pieces a thread
    static constexpr int PPR = T ? ROWS / 8 : 8;                  // pieces per LDS row
    static constexpr int STEP = 256 / PPR;                        // LDS rows from one piece of a thread to its next
    static constexpr int BYTES = ROWS * 128;
    half8_t v[NP];
    const half_t* at[T ? 1 : NP];       // this lane's pieces of slab 0
    int64_t step;                       // T: elements from one piece of a lane to its next
    int32_t left;                       // T: elements of the piece inside its row (8: whole, <= 0: none)
    int pc, lr;

    __device__ __forceinline__ void start(const half_t* base, int32_t r0, int32_t L, int32_t k) {
        pc = threadIdx.x % PPR;
        lr = threadIdx.x / PPR;
        if constexpr (T) {
            left = min(L - r0 - pc * 8, 8);
            at[0] = base + (int64_t)lr * L + r0 + (left > 0 ? pc * 8 : 0);
            step = (int64_t)STEP * L;
        } else {
#pragma unroll
            for (int p = 0; p < NP; ++p) at[p] = base + (int64_t)min(r0 + lr + p * STEP, L - 1) * k + pc * 8;      // (rows past the last are not stored)
        }
    }
    // slab k0 .. k0 + 63 (the pointers move on to the next one); `inside`: it lies inside K and, T, eight rows before its end where the tile reaches past the
    // matrix, whose pieces are read with what lies behind the rows' ends then (it feeds outputs that are not stored) and stay inside the operand.  (Every slab of such a
    // tile under conditions, load by load, took twice as long: 3 entries of 118 x 80 outputs, K = 290, both stored (K, rows), 15.7 us, 5.2 so, 43 of 4 x 118, K = 344 13.7 and 5.2.)
    __device__ __forceinline__ void load(int32_t k0, int32_t k, int32_t L, bool inside) {
        if (inside) {
#pragma unroll
            for (int p = 0; p < NP; ++p) v[p] = load_half8_any(T ? at[0] + p * step : at[p]);
        } else {
            const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
            // whole pieces first, into registers of their own, so that none waits for another
#pragma unroll
            for (int p = 0; p < NP; ++p) v[p] = half8_kept(zero);
            auto have = [&](int p) __attribute__((always_inline)) { return T ? (k0 + lr + p * STEP < k ? left : 0) : k - k0 - pc * 8; };
#pragma unroll
            for (int p = 0; p < NP; ++p)
                if (have(p) >= 8) v[p] = load_half8_any(T ? at[0] + p * step : at[p]);
#pragma unroll
            for (int p = 0; p < NP; ++p)
                if (have(p) > 0 && have(p) < 8) v[p] = load_half8_head_any(T ? at[0] + p * step : at[p], have(p), zero);
        }
        if constexpr (T) {
            at[0] += (int64_t)64 * L;
        } else {
#pragma unroll
            for (int p = 0; p < NP; ++p) at[p] += 64;
        }
    }
    __device__ __forceinline__ void put(int8_t* lds) const {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int r = lr + p * STEP;
            if constexpr (T) *reinterpret_cast<half8_t*>(lds + r * (ROWS * 2) + (((pc >> 1) ^ (r & 3)) << 5) + ((pc & 1) << 4)) = v[p];
            else *reinterpret_cast<half8_t*>(lds + r * 128 + ((pc ^ (r & 7)) << 4)) = v[p];
        }
    }
    // the fragment of block u (16 rows of the tile), k-step ks (32 of K)
    static __device__ __forceinline__ half8_t frag(const int8_t* lds, int u, int ks, int r16, int q) {
        if constexpr (T) {
            typedef short short4_t __attribute__((ext_vector_type(4)));
            const uint32_t p0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const int8_t*)lds + (ks * 32 + q * 8 + (r16 >> 2)) * (ROWS * 2) +
                                ((u ^ (r16 >> 2)) << 5) + ((r16 & 3) << 3);
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)p0);
            const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(uintptr_t)(p0 + 4 * ROWS * 2));
            return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
            return *reinterpret_cast<const half8_t*>(lds + (u * 16 + r16) * 128 + (((ks * 4 + q) ^ (r16 & 7)) << 4));
        }
    }
};

// F32: the sums as they are, straight from the registers (parts of a sum that is not rounded yet, gemm_sum.hip).
template <bool PT, bool QT, int TR, int TC, bool F32 = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TR * TC > 8192 ? 3 : 4))) void k_gemm_any(AnyArgs a) {
    constexpr int WC = TR == 128 ? 2 : 4;                         // waves side by side; each has 64 rows x TC / WC columns
    constexpr int NJ = TC / WC / 16;
    using SP = AnySlab<PT, TR>;
    using SQ = AnySlab<QT, TC>;
    constexpr int OUT = TR * TC * 2, SLABS = SP::BYTES + SQ::BYTES;
    __shared__ __attribute__((aligned(16))) int8_t lds[OUT > SLABS ? OUT : SLABS];
    int8_t* const ldsq = lds + SP::BYTES;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, q = lane >> 4, wr = wave / WC, wc = wave % WC;
    // column tiles of a row of tiles follow one another on one XCD: they share cache lines where rows of the output are not whole ones
    const uint32_t t = a.first + xcd_remap(blockIdx.x, a.tiles);
    const uint32_t b = t / (a.tiles_r * a.tiles_c), rest = t - b * (a.tiles_r * a.tiles_c), tr = rest / a.tiles_c, tc = rest - tr * a.tiles_c;
    // Of an operand stored (K, rows) the last tile lies inside the matrix, if that holds one: what it shares with the one before is computed
    // and stored twice, alike, and no piece crosses a row's end (64 x 300 x 300, 250 tiles 10.3 -> 6.3 us).
    const int32_t j0 = PT && a.n >= TR ? min((int32_t)tr * TR, a.n - TR) : (int32_t)tr * TR, i0 = QT && a.m >= TC ? min((int32_t)tc * TC, a.m - TC) : (int32_t)tc * TC;
    SP sp;
    SQ sq;
    sp.start(a.P + b * a.strideP, j0, a.n, a.k);
    sq.start(a.Q + b * a.strideQ, i0, a.m, a.k);
    const int32_t kp = !PT || j0 + TR <= a.n ? a.k : a.k - 8, kq = !QT || i0 + TC <= a.m ? a.k : a.k - 8;
    auto load = [&](int32_t k0) __attribute__((always_inline)) {
        sp.load(k0, a.k, a.n, k0 + 64 <= kp);
        sq.load(k0, a.k, a.m, k0 + 64 <= kq);
    };
    float4_t acc[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    load(0);
#pragma unroll 1       // (more takes registers that 128 x 128 tiles do not have)
    for (int32_t k0 = 0; k0 < a.k; k0 += 64) {
        if (k0 > 0) __syncthreads();                              // the slab before has been read
        sp.put(lds);
        sq.put(ldsq);
        __syncthreads();
        if (k0 + 64 < a.k) load(k0 + 64);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            half8_t fp[4], fq[NJ];
#pragma unroll
            for (int i = 0; i < 4; ++i) fp[i] = SP::frag(lds, wr * 4 + i, ks, r16, q);
#pragma unroll
            for (int j = 0; j < NJ; ++j) fq[j] = SQ::frag(ldsq, wc * NJ + j, ks, r16, q);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[j], fp[i], acc[i][j], 0, 0, 0);
        }
    }
    if constexpr (F32) {
        struct __attribute__((packed, aligned(8))) Float4Pairs { float4_t v; };      // (m is even)
        struct __attribute__((packed, aligned(8))) Float2 { float x, y; };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t row = j0 + wr * 64 + i * 16 + r16;
            if (row >= a.n) continue;
            float* const dst = static_cast<float*>(a.out) + ((int64_t)b * a.n + row) * a.m;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int32_t col = i0 + (wc * NJ + j) * 16 + q * 4;
                if (col + 4 <= a.m) reinterpret_cast<Float4Pairs*>(dst + col)->v = acc[i][j];
                else if (col < a.m) *reinterpret_cast<Float2*>(dst + col) = Float2{acc[i][j][0], acc[i][j][1]};
            }
        }
        return;
    }
    __syncthreads();
    // Lane l, register e of a 16 x 16 result: output row l % 16, column (l / 16) * 4 + e.  The tile is put together in LDS, piece p of
    // row r at p ^ (r % 8), and leaves in whole rows.
    constexpr int PPO = TC / 8, ROW = TC * 2;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[i][j][e];
            const int piece = (wc * NJ + j) * 2 + (q >> 1);
            *reinterpret_cast<half4_t*>(lds + (wr * 64 + i * 16 + r16) * ROW + ((piece ^ (r16 & 7)) << 4) + ((q & 1) << 3)) = h;
        }
    __syncthreads();
    const int oc = tid % PPO;
    const int32_t left = a.m - i0 - oc * 8;
    half_t* const ob = static_cast<half_t*>(a.out) + ((int64_t)b * a.n + j0) * a.m + i0 + oc * 8;
#pragma unroll
    for (int r = tid / PPO; r < TR; r += 256 / PPO) {
        if (j0 + r >= a.n || left <= 0) continue;
        const half8_t h = *reinterpret_cast<const half8_t*>(lds + r * ROW + ((oc ^ (r & 7)) << 4));
        half_t* const dst = ob + (int64_t)r * a.m;
        if (left >= 8) store_half8_any(dst, h);
        else store_half8_head_any(dst, left, h);
    }
}

// 0 or an error code.  A (batchA, k, m) [(batchA, m, k) if aT], B (batchB, n, k) [(batchB, k, n) if bT], out (batch, n, m); f32 (operands stored (K, rows)): fp32 out.
int gemm_f16_any(int32_t m, int32_t k, int32_t n, int32_t batchA, int32_t batchB, int aT, int bT, const void* A, const void* B, void* out, hipStream_t st, bool f32) {
    AnyArgs a;
    a.P = (const half_t*)B; a.Q = (const half_t*)A; a.out = out;
    a.strideP = batchB == 1 ? 0 : (int64_t)n * k;
    a.strideQ = batchA == 1 ? 0 : (int64_t)m * k;
    a.n = n; a.m = m; a.k = k;
    const int64_t batch = batchA > batchB ? batchA : batchB;
    // tiles of 128 rows or columns unless they cover a quarter more than those of 64
    auto wide = [](int64_t len) { return ceil_div(len, 128) * 128 * 4 <= ceil_div(len, 64) * 64 * 5; };
    // ... and small ones where those are at most one a compute unit: a slab of them is there sooner (over 490 such products a tenth quicker, none slower)
    const bool few = ceil_div(n, 64) * ceil_div(m, 64) * batch <= compute_units();
    const bool wr = wide(n) && !few, wc = wide(m) && !few;
    const int64_t tr = ceil_div(n, wr ? 128 : 64), tc = ceil_div(m, wc ? 128 : 64), total = tr * tc * batch;
    a.tiles_r = (uint32_t)tr; a.tiles_c = (uint32_t)tc;
    if (total >= 1ll << 32) return CPMK_ETOOBIG;
    for (int64_t t0 = 0; t0 < total; t0 += 1 << 23) {       // (a launch holds fewer than 2^32 threads)
        a.first = (uint32_t)t0;
        a.tiles = (uint32_t)(total - t0 < 1 << 23 ? total - t0 : 1 << 23);
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(a.tiles), dim3(256), 0, st, a); };
        auto pick = [&](auto pt, auto qt, auto fc) {
            constexpr bool PT = decltype(pt)::value, QT = decltype(qt)::value, F = decltype(fc)::value;
            if (wr) wc ? go(k_gemm_any<PT, QT, 128, 128, F>) : go(k_gemm_any<PT, QT, 128, 64, F>);
            else wc ? go(k_gemm_any<PT, QT, 64, 128, F>) : go(k_gemm_any<PT, QT, 64, 64, F>);
        };
        if (f32) pick(std::true_type{}, std::true_type{}, std::true_type{});
        else if (!bT) aT ? pick(std::false_type{}, std::false_type{}, std::false_type{}) : pick(std::false_type{}, std::true_type{}, std::false_type{});
        else aT ? pick(std::true_type{}, std::false_type{}, std::false_type{}) : pick(std::true_type{}, std::true_type{}, std::false_type{});
        if (const int e = launch_status()) return e;
    }
    return 0;
}

}  // namespace cpmk
