// Backward pass of the normalisation over dim 1 with its affine coefficients, from the fp32 statistics that the
// forward pass kept:  with  xh = (x - mean) * rstd  and  gw = grad * alpha
//     grad_x = rstd * ( gw - sum_i(gw) / n - xh * sum_i(gw * xh) / n )        (without a mean: no first sum)
//     grad_alpha[i] = sum_{b,j} grad * xh,     grad_beta[i] = sum_{b,j} grad
// The reference recomputes the normalised tensor and its statistics and walks the tensors five times
// (cpm_kernels/torch/layernorm.py:31-86, 113-156; cuda/layernorm.cu:142-339, cuda/arith.cu:213-330).
//
// Bound by memory: x and grad in, grad_x out, once each.  The column tile of dim1.h (64 columns x 256 rows of both
// inputs in registers, 512 rows beyond 8192; taller columns in teams), whose rows' sums over its 64 columns leave as fp32 partials that a second small
// kernel adds up in a fixed order.  8 x 4096 x 512: 82 us in five kernels and ten passes before, now 31 + 5 us
// (3.2 TB/s; with 512 rows a part and one workgroup a compute unit 33; 16 x 4096 x 1024: 114, 119).
#include "dim1.h"
#include "exchange.h"
#include <type_traits>

namespace cpmk {

struct LnBwdArgs {
    int32_t n, m;
    const half_t* x;
    const half_t* g;
    const half_t* alpha;       // (n)
    const float* stats;        // (batch, 2, m): mean, rstd
    half_t* out;               // grad_x
    float* part;               // (batch * tiles, 2, n): a tile's row sums of grad and of grad * xh
};

// v added over the eight lanes that share lane / 8
__device__ __forceinline__ float lanes_div8_sum(float v) {
    auto dpp = [](float x, auto c) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(c)::value, 0xf, 0xf, true));
    };
    v += dpp(v, std::integral_constant<int, 0xB1>{});       // quad_perm [1,0,3,2]
    v += dpp(v, std::integral_constant<int, 0x4E>{});       // quad_perm [2,3,0,1]
    return v + dpp(v, std::integral_constant<int, 0x141>{});      // row_half_mirror
}

// MODE as in train.hip's k_col_team: 0 non-temporal 16-byte accesses, 1 plain ones, 2 any width and alignment.
// (R = 4: two 512-thread workgroups share a compute unit, at most 128 registers per lane, so the products of the sums are not
// kept for the outputs but formed again)
template <int R, int MODE, bool MEAN>
__global__ __launch_bounds__(512, R == 4 ? 4 : 2) void k_ln_bwd_team(LnBwdArgs p, int32_t tiles_per_batch, int32_t parts,
                                                                                                uint32_t nteams, XchLaunch xl) {
    constexpr int NT = 512, LPR = 8, NV = MEAN ? 2 : 1;
    constexpr bool NTH = MODE == 0, UA = MODE == 2;
    using T = ColTile<NT, LPR, R>;
    __shared__ float lds[(T::NW + 1) * T::COLS * NV];
    __shared__ float tot[T::COLS * NV];
    const int tid = threadIdx.x, cg = tid % LPR, rg = tid / LPR;
    XchMember me;
    if (!xch_member(blockIdx.x, parts, nteams, me)) return;
    const uint32_t part = me.part, team = me.team;
    const uint32_t b = team / tiles_per_batch, ct = team - b * tiles_per_batch;
    const int32_t col0 = ct * T::COLS + cg * 8;
    const int32_t own0 = part * T::ROWS, own_n = min(T::ROWS, p.n - own0);
    const int64_t boff = (int64_t)b * p.n * p.m + (int64_t)own0 * p.m;

    // what the sums need besides the tiles, requested ahead of them (loads return in order)
    half_t w[R];
#pragma unroll
    for (int q = 0; q < R; ++q) w[q] = p.alpha[min(own0 + q * T::RPP + rg, p.n - 1)];
    float rstd[8], shift[8];        // xh = x * rstd + shift
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int32_t c = min(col0 + e, p.m - 1);
        rstd[e] = p.stats[((int64_t)b * 2 + 1) * p.m + c];
        shift[e] = MEAN ? -p.stats[(int64_t)b * 2 * p.m + c] * rstd[e] : 0.0f;
    }
    half8_t vx[R], vg[R];
    constexpr int LOADS = UA ? kLoadsUnset : R == 8 || MEAN ? kLoadsPlain : kLoadsKept;        // (128 registers hold four rows and means only so)
    coltile_request<NT, LPR, R, NTH, UA, LOADS>(vg, p.g + boff, own_n, p.m, col0, (half_t)0.0f);
    coltile_request<NT, LPR, R, NTH, UA, LOADS>(vx, p.x + boff, own_n, p.m, col0, (half_t)0.0f);
    coltile_settle<NT, LPR, R, UA, LOADS>(vg, own_n, p.m, col0, (half_t)0.0f);
    coltile_settle<NT, LPR, R, UA, LOADS>(vx, own_n, p.m, col0, (half_t)0.0f);
    float* const prow = p.part + ((int64_t)team * 2 + (cg & 1)) * p.n + own0;
    float s[NV * 8];
#pragma unroll
    for (int e = 0; e < NV * 8; ++e) s[e] = 0.0f;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const float a = (float)w[q];
        float r0 = 0.0f, r1 = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float gi = (float)vg[q][e], gx = gi * __builtin_fmaf((float)vx[q][e], rstd[e], shift[e]);      // (elements past an edge: grad is zero)
            if constexpr (MEAN) {
                s[8 + e] += gi * a;
                r0 += gi;
            }
            s[e] += gx * a;
            r1 += gx;
        }
        if constexpr (MEAN) r0 = lanes_div8_sum(r0);
        r1 = lanes_div8_sum(r1);
        const int32_t lrow = q * T::RPP + rg;
        if (cg < 2 && lrow < own_n && (MEAN || cg == 1)) prow[lrow] = cg == 0 ? r0 : r1;
        __builtin_amdgcn_sched_barrier(0);       // a row at a time: interleaving all of them costs registers
    }
    if (parts == 1) {
        coltile_reduce<NT, LPR, NV, false>(s, lds);
    } else {
        uint64_t* team_slots = xl.region + (size_t)team * parts * kXchVals;
        coltile_reduce_to<NT, LPR, NV, false>(s, lds, [&](int i, float r) { xch_post(team_slots + (size_t)part * kXchVals, i, r, xl.tag); });
        if (tid < T::COLS * NV) {
            const uint64_t deadline = wall_clock64() + kXchTimeoutTicks;
            float acc = 0.0f;
            bool ok = true;
            for (int32_t q0 = 0; q0 < parts; q0 += 4) {
                float v[4];
                ok &= xch_gather<4>(team_slots, parts, q0, tid, xl.tag, deadline, v);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc += v[j];       // part order; absent parts are zeros
            }
            tot[tid] = ok ? acc : __builtin_nanf("");
            if (!ok) xch_flag(xl, kXchStatusTimeout);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NV * 8; ++e) s[e] = tot[(e >> 3) * T::COLS + cg * 8 + (e & 7)];
    }
    const float rn = 1.0f / (float)p.n;
    // grad_x = rstd * gw - x * (rstd * rstd * s0 / n) - (rstd * (shift * s0 + s1) / n):  three constants per column
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float k = s[e] * rn * rstd[e];
        shift[e] = MEAN ? __builtin_fmaf(shift[e], k, s[(MEAN ? 8 : 0) + e] * rn * rstd[e]) : 0.0f;
        s[e] = k * rstd[e];
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
        int4_t xi = __builtin_bit_cast(int4_t, vx[q]), gi4 = __builtin_bit_cast(int4_t, vg[q]);
        asm volatile("" : "+v"(xi), "+v"(gi4));         // (the conversions of the sums are not kept for here)
        const half8_t xh = __builtin_bit_cast(half8_t, xi), gh = __builtin_bit_cast(half8_t, gi4);
        const float a = (float)w[q];
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float gw = (float)gh[e] * a;
            o[e] = (half_t)__builtin_fmaf(-(float)xh[e], s[e], MEAN ? __builtin_fmaf(gw, rstd[e], -shift[e]) : gw * rstd[e]);
        }
        vx[q] = o;
        __builtin_amdgcn_sched_barrier(0);
    }
    coltile_store<NT, LPR, R, NTH, UA>(vx, p.out + boff, own_n, p.m, col0);
    if (parts > 1 && tid < 64) xch_retire(xl, team, parts);
}

// grad_alpha / grad_beta[i] = sum over the tiles of their partial row sums, in a fixed order: 64 rows x 4 groups of tiles
// per workgroup, blockIdx.y the kind (0 grad, 1 grad * xh).
__global__ __launch_bounds__(256) void k_ln_param_sum(int32_t n, int32_t tiles, int first, const float* __restrict__ part, half_t* grad_alpha,
                                                      half_t* grad_beta) {
    __shared__ float red[4][64];
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6, kind = blockIdx.y + first;
    const int32_t i = blockIdx.x * 64 + c;
    float s = 0.0f;
    if (i < n) {
        for (int32_t t0 = rg; t0 < tiles; t0 += 32) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = t0 + u * 4 < tiles ? part[((int64_t)(t0 + u * 4) * 2 + kind) * n + i] : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
    }
    red[rg][c] = s;
    __syncthreads();
    if (rg == 0 && i < n) (kind ? grad_alpha : grad_beta)[i] = (half_t)((red[0][c] + red[1][c]) + (red[2][c] + red[3][c]));
}

// Columns taller than a team holds, or launches recorded when no packets are left: both passes through memory, 64 columns x 4
// row groups per workgroup; the row sums of the tile by the workgroup's first 64 lanes' neighbours (lane = column).
template <bool MEAN>
__global__ __launch_bounds__(256) void k_ln_bwd_any(LnBwdArgs p, int32_t tiles_per_batch) {
    __shared__ float red[2][4][64];
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const int64_t tile = blockIdx.x, b = tile / tiles_per_batch;
    const int32_t col = (int32_t)(tile - b * tiles_per_batch) * 64 + c, n = p.n, m = p.m;
    const int64_t boff = b * n * m;
    const bool live = col < m;
    const float mean = MEAN && live ? p.stats[b * 2 * m + col] : 0.0f, rstd = live ? p.stats[(b * 2 + 1) * m + col] : 0.0f;
    float s0 = 0.0f, s1 = 0.0f;
    for (int32_t i = rg; i < n; i += 4) {
        const float g = live ? (float)p.g[boff + (int64_t)i * m + col] : 0.0f;
        const float gx = live ? g * (((float)p.x[boff + (int64_t)i * m + col] - mean) * rstd) : 0.0f;
        const float a = (float)p.alpha[i];
        s0 += gx * a;
        s1 += g * a;
        const float r0 = wave_sum(g), r1 = wave_sum(gx);
        if (c == 0) {
            if (MEAN) p.part[(tile * 2) * n + i] = r0;
            p.part[(tile * 2 + 1) * n + i] = r1;
        }
    }
    red[0][rg][c] = s0;
    red[1][rg][c] = s1;
    __syncthreads();
    s0 = (red[0][0][c] + red[0][1][c] + red[0][2][c] + red[0][3][c]) / (float)n;
    s1 = MEAN ? (red[1][0][c] + red[1][1][c] + red[1][2][c] + red[1][3][c]) / (float)n : 0.0f;
    if (!live) return;
    for (int32_t i = rg; i < n; i += 4) {
        const int64_t o = boff + (int64_t)i * m + col;
        const float gw = (float)p.g[o] * (float)p.alpha[i];
        p.out[o] = (half_t)(rstd * (gw - s1 - (((float)p.x[o] - mean) * rstd) * s0));
    }
}

static int ln_bwd(int32_t batch, const LnBwdArgs& p, bool mean, hipStream_t st) {
    constexpr int64_t kMaxParts = 32;
    // 256 rows a part, two workgroups a compute unit (their loads and stores pass under each other's sums); 512 rows, one
    // workgroup, where the team would be too large
    const int64_t rows = p.n <= 256 * kMaxParts ? 256 : 512;
    const int64_t tiles = ceil_div(p.m, 64), parts = ceil_div(p.n, rows);
    const bool vec16 = p.m % 8 == 0 && aligned16(p.x) && aligned16(p.g) && aligned16(p.out);
    auto on_line = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 127u) == 0; };
    const bool lines = vec16 && p.m % 64 == 0 && on_line(p.x) && on_line(p.g) && on_line(p.out);
    if ((int64_t)p.n * p.m < (1ll << 31) && parts <= kMaxParts && tiles * parts <= kXchSlots) {
        // one packet slot per (team, part): batches beyond the pool go out in several launches
        const int64_t per_launch = parts > 1 ? kXchSlots / (tiles * parts) : ((1ll << 31) - 8) / (tiles * parts);
        bool no_slots = false;
        for (int64_t b0 = 0; b0 < batch; b0 += per_launch) {
            const int64_t nb = batch - b0 < per_launch ? batch - b0 : per_launch;
            LnBwdArgs q = p;
            q.x += b0 * p.n * p.m; q.g += b0 * p.n * p.m; q.out += b0 * p.n * p.m;
            q.stats += b0 * 2 * p.m; q.part += b0 * tiles * 2 * p.n;
            XchScope xs;
            if (parts > 1) {
                const int rc = xs.begin(tiles * nb * parts, st);
                if (rc == kXchFull && b0 == 0) {
                    no_slots = true;
                    break;
                }
                if (rc != 0) return rc == kXchFull ? CPMK_ETOOBIG : rc;
            }
            auto go = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3((unsigned)xch_team_grid(tiles * nb, parts)), dim3(512), 0, st, q, (int32_t)tiles, (int32_t)parts,
                                   (uint32_t)(tiles * nb), xs.xl);
            };
            auto pick = [&](auto rc, auto mc) {
                constexpr int R = decltype(rc)::value;
                constexpr bool MEAN = decltype(mc)::value;
                if (!vec16) go(k_ln_bwd_team<R, 2, MEAN>);
                else if (lines) go(k_ln_bwd_team<R, 0, MEAN>);
                else go(k_ln_bwd_team<R, 1, MEAN>);
            };
            using R4 = std::integral_constant<int, 4>;
            using R8 = std::integral_constant<int, 8>;
            if (rows == 256) { if (mean) pick(R4{}, std::true_type{}); else pick(R4{}, std::false_type{}); }
            else { if (mean) pick(R8{}, std::true_type{}); else pick(R8{}, std::false_type{}); }
            const int e = launch_status();
            const int rc2 = xs.end();
            if (e != 0 || rc2 != 0) return e ? e : rc2;
        }
        if (!no_slots) return 0;
    }
    if (!grid_fits(tiles * batch)) return CPMK_ETOOBIG;
    if (mean) hipLaunchKernelGGL(k_ln_bwd_any<true>, dim3((unsigned)(tiles * batch)), dim3(256), 0, st, p, (int32_t)tiles);
    else hipLaunchKernelGGL(k_ln_bwd_any<false>, dim3((unsigned)(tiles * batch)), dim3(256), 0, st, p, (int32_t)tiles);
    return launch_status();
}

}  // namespace cpmk

using namespace cpmk;

extern "C" {

int cpmk_layernorm_affine_backward(int32_t batch, int32_t n, int32_t m, const void* mat, const void* grad_out, const void* alpha,
                                   const void* stats, void* grad, void* grad_alpha, void* grad_beta, void* partials, void* stream) {
    clear_stale_error();
    if (batch < 0 || n < 0 || m < 0) return CPMK_EBADARG;
    if ((int64_t)batch * n * m == 0) return 0;
    if (any_null(mat, grad_out, alpha, stats, grad, grad_alpha, partials)) return CPMK_EBADARG;
    const int64_t tiles = ceil_div(m, 64) * batch;
    if (tiles > 0x3fffffff) return CPMK_ETOOBIG;
    const bool mean = grad_beta != nullptr;
    const LnBwdArgs p = {n, m, (const half_t*)mat, (const half_t*)grad_out, (const half_t*)alpha, (const float*)stats, (half_t*)grad, (float*)partials};
    if (int e = ln_bwd(batch, p, mean, (hipStream_t)stream)) return e;
    hipLaunchKernelGGL(k_ln_param_sum, dim3((unsigned)ceil_div(n, 64), mean ? 2 : 1), dim3(256), 0, (hipStream_t)stream, n, (int32_t)tiles, mean ? 0 : 1,
                       (const float*)partials, (half_t*)grad_alpha, (half_t*)grad_beta);
    return launch_status();
}

}  // extern "C"
