// Gradient of a token embedding's table from gradient rows (tokens, hidden): row v is the fp32 sum of the rows of the
// tokens with id v (what the two stages of cuda/embedding.cu:36-88 compute together), rounded once.
//   k_rank_ids         the tokens in the order of their ids (equal ids in the order of the tokens)
//   k_embedding_pieces sums of the runs of equal ids inside pieces of 32 sorted tokens; runs that lie inside a piece are
//                      rows of the gradient, what crosses a piece's edge is left as fp32 partial sums
//   k_embedding_runs   partial sums of a run that crosses edges -> its row
// The order of every sum is fixed by the ids alone.  Rows of ids that do not occur are not written (the caller clears them).
#include "common.h"

namespace cpmk {

// A token's rank is the number of ids that sort before its own, counted outright: a workgroup takes 64 tokens, one per
// lane, and its 16 waves a sixteenth of the ids each, which reach a wave as scalars (two vector operations per id and 64
// tokens).  One launch and no scratch where a radix sort takes several of each.
constexpr int kRankWaves = 16;
__device__ __forceinline__ void rank_ids(uint32_t block, int32_t tokens, const int32_t* __restrict__ ids, int32_t* __restrict__ order,
                                         int32_t* __restrict__ sorted) {
    __shared__ int32_t part[kRankWaves][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int32_t p0 = block * 64, p = p0 + lane;
    const int32_t id = ids[min(p, tokens - 1)];
    const int32_t share = (tokens + kRankWaves - 1) / kRankWaves;
    const int32_t q0 = min(wave * share, tokens), q1 = min(q0 + share, tokens);
    int32_t before = 0;
    // the ids of earlier tokens come before an equal one, those of later tokens do not; the 64 tokens themselves lie between
    const int32_t e1 = min(q1, p0), e2 = min(q1, p0 + 64);
#pragma unroll 16
    for (int32_t q = q0; q < e1; ++q) before += ids[q] <= id ? 1 : 0;
    for (int32_t q = max(q0, p0); q < e2; ++q) before += (ids[q] < id || (ids[q] == id && q < p)) ? 1 : 0;
#pragma unroll 16
    for (int32_t q = max(q0, p0 + 64); q < q1; ++q) before += ids[q] < id ? 1 : 0;
    part[wave][lane] = before;
    __syncthreads();
    if (wave == 0 && p < tokens) {
        int32_t rank = 0;
#pragma unroll
        for (int w = 0; w < kRankWaves; ++w) rank += part[w][lane];
        order[rank] = p;
        sorted[rank] = id;
    }
}

__global__ __launch_bounds__(64 * kRankWaves) void k_rank_ids(int32_t tokens, const int32_t* __restrict__ ids, int32_t* __restrict__ order,
                                                              int32_t* __restrict__ sorted) {
    rank_ids(blockIdx.x, tokens, ids, order, sorted);
}

// What has to be done before the rows are summed, in one launch: the order of the ids, the gradient (batch, hidden, seq) as rows (tokens, hidden),
// and zeros in the table.  Bound by memory: the counting, 64 workgroups that hardly use it, and the transposition, which waits at barriers, pass under
// the zeros: 4096 tokens x 4096 beside 30000 rows 64 us in three launches, 42 so; 310 x 1216 beside 11794 12.1 and 7.3; 16384 x 2048 beside 50000, where the
// counting takes 24, 92 and 48.
struct PrepareArgs {
    int32_t tokens, hidden, seq;
    const half_t* grad;
    half_t *rows, *table;
    int64_t total;                // elements of the table
    uint32_t rank_blocks, tile_blocks, tiles_c, tiles_r, tiles;
    uint32_t first;               // number of the launch's first workgroup
};
constexpr int kPrepareThreads = 64 * kRankWaves;
constexpr int64_t kFillBytes = 8 * 16 * kPrepareThreads;      // zeros a workgroup writes

// PIECES: rows of grad and of the transposed rows are whole aligned 16-byte pieces: a wave transposes a tile of 64 x 64 in registers, each
// lane a block of 8 x 8, with 128-byte segments on both sides; else through LDS.
// (the ids are an argument of their own, which no other pointer reaches: as a member of `a` the compiler took their loads for ones that the stores here
// could change and left them to the vector unit, sixteen ids four vector loads instead of one scalar one: 250 x 64 tokens of 70 beside 500 rows 38.1 us, 24.2 so)
template <bool PIECES>
__global__ __launch_bounds__(kPrepareThreads) void k_embedding_prepare(PrepareArgs a, const int32_t* __restrict__ ids, int32_t* __restrict__ order,
                                                                       int32_t* __restrict__ sorted) {
    const uint32_t wg = a.first + blockIdx.x;
    if (wg < a.rank_blocks) {
        rank_ids(wg, a.tokens, ids, order, sorted);
        return;
    }
    const uint32_t at = wg - a.rank_blocks;
    const bool is_tile = at < a.tile_blocks;
    const uint32_t block = is_tile ? at : at - a.tile_blocks;
    if (is_tile) {
        const int32_t n = a.hidden, m = a.seq;
        const uint32_t per = a.tiles_c * a.tiles_r;
        if constexpr (PIECES) {
            const uint32_t t = block * kRankWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            if (t >= a.tiles) return;
            const uint32_t b = t / per, in = t - b * per, tr = in / a.tiles_c, tc = in - tr * a.tiles_c;
            const int64_t boff = (int64_t)b * n * m;
            const int lane = threadIdx.x & 63;
            half8_t v[8];
            {
                const int32_t r = tr * 64 + (lane >> 3) * 8, c = tc * 64 + (lane & 7) * 8;
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    v[p] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
                    if (r < n && c < m) v[p] = __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(a.grad + boff + (int64_t)(r + p) * m + c));
                }
            }
            transpose_half8x8(v);
            // (lane l has block (l / 8, l % 8): what it stores lies beside what the lanes eight apart do)
            const int32_t r = tr * 64 + (lane >> 3) * 8, c = tc * 64 + (lane & 7) * 8;
            if (r < n && c < m)
#pragma unroll
                for (int e = 0; e < 8; ++e) *reinterpret_cast<half8_t*>(a.rows + boff + (int64_t)(c + e) * n + r) = v[e];
        } else {
            // four tiles of 64 x 64, 256 lanes each
            __shared__ __attribute__((aligned(16))) TransposeTile tile[4];
            const int sub = threadIdx.x >> 8, tid = threadIdx.x & 255;
            const uint32_t t = block * 4 + sub;
            const uint32_t b = t / per, in = t - b * per, tr = in / a.tiles_c, tc = in - tr * a.tiles_c;
            const int32_t r0 = tr * 64, c0 = tc * 64, rows = t < a.tiles ? n : 0;
            const int64_t boff = (int64_t)b * n * m;
            transpose_tile_in(tile[sub], a.grad + boff, rows, m, r0, c0, tid);
            __syncthreads();
            if (rows) transpose_tile_out(tile[sub], a.rows + boff, n, m, r0, c0, tid);
        }
        return;
    }
    const int64_t pieces = a.total >> 3, p0 = (int64_t)block * (kFillBytes / 16) + threadIdx.x;
    half8_t* const table = reinterpret_cast<half8_t*>(a.table);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int64_t p = p0 + u * kPrepareThreads;
        if (p < pieces) table[p] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
    if (block == 0 && threadIdx.x < (a.total & 7)) a.table[(pieces << 3) + threadIdx.x] = (half_t)0.0f;
}

// Sorted tokens a workgroup sums up.  Thirty-two rows hide the latency of the gather (all are requested before the first is
// added) and split even one id's thousands of tokens over many workgroups.
constexpr int kPiece = 32;

// VEC halves at a time: 8 where rows are whole 16-byte pieces, else 1.
template <int VEC>
struct RowPiece {
    half_t h[VEC];
};
template <int VEC>
__device__ __forceinline__ RowPiece<VEC> row_load(const half_t* p) {
    RowPiece<VEC> r;
    if constexpr (VEC == 8) {
        const half8_t v = *reinterpret_cast<const half8_t*>(p);
#pragma unroll
        for (int e = 0; e < 8; ++e) r.h[e] = v[e];
    } else {
        r.h[0] = *p;
    }
    return r;
}
template <int VEC>
__device__ __forceinline__ void row_store(half_t* p, const float (&s)[VEC]) {
    if constexpr (VEC == 8) {
        half8_t v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = round_f16(s[e]);
        *reinterpret_cast<half8_t*>(p) = v;
    } else {
        *p = round_f16(s[0]);
    }
}

// Bound by the gather of `rows`, which was written just before and is read from the last-level cache (4096 tokens x 4096: 15 us, and 4 us for
// the runs; the two stages that walk a batch entry's tokens in one chain 82 + 6 us).  Partial sums of
// piece c: row 2c the run that began before the piece, row 2c + 1 the run that begins in it and goes on behind it.
template <int VEC>
__global__ __launch_bounds__(256) void k_embedding_pieces(int32_t tokens, int32_t hidden, const half_t* __restrict__ rows,
                                                          const int32_t* __restrict__ order, const int32_t* __restrict__ sorted,
                                                          half_t* __restrict__ grad, float* __restrict__ partials) {
    const int32_t c = blockIdx.x, p0 = c * kPiece, p1 = min(p0 + kPiece, tokens);
    const int32_t col = (blockIdx.y * 256 + threadIdx.x) * VEC;
    if (col >= hidden) return;
    bool head = p0 > 0 && sorted[p0 - 1] == sorted[p0];
    const bool goes_on = p1 < tokens && sorted[p1 - 1] == sorted[p1];
    float s[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) s[e] = 0.0f;
    constexpr int U = 16;
#pragma unroll
    for (int u0 = 0; u0 < kPiece; u0 += U) {
        RowPiece<VEC> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = row_load<VEC>(rows + (int64_t)order[min(p0 + u0 + u, p1 - 1)] * hidden + col);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t p = p0 + u0 + u;
            if (p >= p1) break;
#pragma unroll
            for (int e = 0; e < VEC; ++e) s[e] += (float)v[u].h[e];
            const bool end = p + 1 == p1;
            if (!end && sorted[p] == sorted[p + 1]) continue;
            if (head || (end && goes_on)) {
                float* dst = partials + ((int64_t)2 * c + (head ? 0 : 1)) * hidden + col;
#pragma unroll
                for (int e = 0; e < VEC; ++e) dst[e] = s[e];
            } else {
                row_store<VEC>(grad + (int64_t)sorted[p] * hidden + col, s);
            }
            head = false;
#pragma unroll
            for (int e = 0; e < VEC; ++e) s[e] = 0.0f;
        }
    }
}

// Piece c's workgroups finish the run that begins in piece c and goes on behind it, if there is one.
template <int VEC>
__global__ __launch_bounds__(256) void k_embedding_runs(int32_t tokens, int32_t hidden, const int32_t* __restrict__ sorted, half_t* __restrict__ grad,
                                                        const float* __restrict__ partials) {
    const int32_t c = blockIdx.x, p0 = c * kPiece, p1 = p0 + kPiece;
    if (p1 >= tokens) return;
    const int32_t id = sorted[p1 - 1];
    if (sorted[p1] != id || (p0 > 0 && sorted[p0 - 1] == id)) return;       // (the second: the run began before this piece)
    // the pieces that the run covers up to their end, 64 looked at together
    const int lane = threadIdx.x & 63;
    int32_t last = c + 1;      // the run's last piece
    for (;;) {
        const int64_t next = ((int64_t)last + lane + 1) * kPiece;         // first token behind piece last + lane
        const uint64_t stops = __builtin_amdgcn_ballot_w64(next >= tokens || sorted[min(next, (int64_t)tokens - 1)] != id);
        if (stops != 0) {
            last += __builtin_ctzll(stops);
            break;
        }
        last += 64;
    }
    const int32_t col = (blockIdx.y * 256 + threadIdx.x) * VEC;
    if (col >= hidden) return;
    float s[VEC];
    const float* first = partials + ((int64_t)2 * c + 1) * hidden + col;
#pragma unroll
    for (int e = 0; e < VEC; ++e) s[e] = first[e];
#pragma unroll 4
    for (int32_t d = c + 1; d <= last; ++d) {
        const float* src = partials + (int64_t)2 * d * hidden + col;
#pragma unroll
        for (int e = 0; e < VEC; ++e) s[e] += src[e];
    }
    row_store<VEC>(grad + (int64_t)id * hidden + col, s);
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_embedding_order_ids(int32_t tokens, const void* ids, void* order, void* sorted_ids, void* stream) {
    clear_stale_error();
    if (tokens < 0) return CPMK_EBADARG;
    if (tokens == 0) return 0;
    if (any_null(ids, order, sorted_ids)) return CPMK_EBADARG;
    hipLaunchKernelGGL(k_rank_ids, dim3((unsigned)ceil_div(tokens, 64)), dim3(64 * kRankWaves), 0, (hipStream_t)stream, tokens, (const int32_t*)ids,
                       (int32_t*)order, (int32_t*)sorted_ids);
    return launch_status();
}

int cpmk_embedding_backward_rows(int32_t tokens, int32_t hidden_size, const void* grad_rows, const void* order, const void* sorted_ids, void* grad,
                                 void* partials, void* stream) {
    clear_stale_error();
    if (tokens < 0 || hidden_size < 0) return CPMK_EBADARG;
    if ((int64_t)tokens * hidden_size == 0) return 0;
    if (any_null(grad_rows, order, sorted_ids, grad, partials)) return CPMK_EBADARG;
    const int64_t pieces = ceil_div(tokens, kPiece);
    auto go = [&](auto vc) {
        constexpr int VEC = decltype(vc)::value;
        const dim3 grid((unsigned)pieces, (unsigned)ceil_div(hidden_size, 256 * VEC));
        hipLaunchKernelGGL((k_embedding_pieces<VEC>), grid, dim3(256), 0, (hipStream_t)stream, tokens, hidden_size, (const half_t*)grad_rows,
                           (const int32_t*)order, (const int32_t*)sorted_ids, (half_t*)grad, (float*)partials);
        if (int e = launch_status()) return e;
        hipLaunchKernelGGL((k_embedding_runs<VEC>), grid, dim3(256), 0, (hipStream_t)stream, tokens, hidden_size, (const int32_t*)sorted_ids,
                           (half_t*)grad, (const float*)partials);
        return launch_status();
    };
    if (ceil_div(hidden_size, 256) > 65535) return CPMK_ETOOBIG;
    if (hidden_size % 8 == 0 && aligned16(grad_rows) && aligned16(grad)) return go(std::integral_constant<int, 8>{});
    return go(std::integral_constant<int, 1>{});
}

int cpmk_embedding_backward_prepare(int32_t batch, int32_t hidden_size, int32_t seq_len, int32_t vocab_size, const void* ids, void* order, void* sorted_ids,
                                    const void* grad_out, void* grad_rows, void* grad, void* stream) {
    clear_stale_error();
    if (batch < 0 || hidden_size < 0 || seq_len < 0 || vocab_size < 0) return CPMK_EBADARG;
    const int64_t tokens = (int64_t)batch * seq_len, total = (int64_t)vocab_size * hidden_size;
    if (tokens >= 1ll << 31) return CPMK_ETOOBIG;
    if ((total > 0 && grad == nullptr) || (tokens * hidden_size > 0 && any_null(grad_out, grad_rows)) || (tokens > 0 && ids && any_null(order, sorted_ids))) return CPMK_EBADARG;
    if (total > 0 && !aligned16(grad)) return CPMK_EALIGN;
    PrepareArgs a;
    a.tokens = (int32_t)tokens; a.hidden = hidden_size; a.seq = seq_len;
    a.grad = (const half_t*)grad_out; a.rows = (half_t*)grad_rows; a.table = (half_t*)grad; a.total = total;
    const bool pieces = hidden_size % 8 == 0 && seq_len % 8 == 0 && aligned16(grad_out) && aligned16(grad_rows);
    const int64_t tc = ceil_div(seq_len, 64), tr = ceil_div(hidden_size, 64), tiles = tc * tr * batch;
    const int64_t rank = ids ? ceil_div(tokens, 64) : 0, tile_blocks = ceil_div(tiles, pieces ? kRankWaves : 4), fill = ceil_div(total * 2, kFillBytes);
    const int64_t total_blocks = rank + tile_blocks + fill;
    if (tiles >= 1ll << 32 || total_blocks >= 1ll << 32) return CPMK_ETOOBIG;       // (more than the device's memory holds)
    a.rank_blocks = (uint32_t)rank; a.tile_blocks = (uint32_t)tile_blocks; a.tiles_c = (uint32_t)tc; a.tiles_r = (uint32_t)tr; a.tiles = (uint32_t)tiles;
    // a launch holds fewer than 2^32 threads: many short sequences, each a tile and more, go out in several
    constexpr int64_t most = (1ll << 32) / kPrepareThreads - 1;
    for (int64_t b0 = 0; b0 < total_blocks; b0 += most) {
        a.first = (uint32_t)b0;
        const dim3 grid((unsigned)(total_blocks - b0 < most ? total_blocks - b0 : most));
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(kPrepareThreads), 0, (hipStream_t)stream, a, (const int32_t*)ids, (int32_t*)order, (int32_t*)sorted_ids);
        };
        if (pieces) go(k_embedding_prepare<true>);
        else go(k_embedding_prepare<false>);
        if (const int e = launch_status()) return e;
    }
    return 0;
}

}  // extern "C"
