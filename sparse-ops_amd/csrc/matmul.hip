// so_matmul: Y[m x C] = act(E * X[n x C] + bias) on gfx950.
//
// One wavefront owns one ELLPACK row and one tile of 64*VEC dense columns.  The
// row's weights and column indices are wave-uniform, so they are fetched with
// scalar loads into SGPRs; every gathered X row segment X[j, c0 .. c0+64*VEC) is
// one fully coalesced vector load; each lane keeps VEC fp32 accumulators that
// start at bias[i] and receive one fused multiply-add per stored nonzero in
// ascending slot order -- the rounding sequence of the reference's inner loop
// (src/ellpack_matmul.cpp:51-66) -- followed by the fused epilogue.
//
// Workgroups are numbered so that each of the 8 XCDs (workgroup id modulo 8)
// works on as few column tiles as possible: an XCD's L2 then has to hold only
// its own tiles' slice of X.
#include "so_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace {

constexpr int kWavesPerGroup = 4;

template <int VEC> struct VecT;
template <> struct VecT<1> { using type = float; };
template <> struct VecT<2> { using type = float2; };
template <> struct VecT<4> { using type = float4; };

template <int VEC>
__device__ __forceinline__ void load_vec(const float *p, float (&v)[VEC])
{
    using T = typename VecT<VEC>::type;
    const T t = *reinterpret_cast<const T *>(p);
    if constexpr (VEC == 1) { v[0] = t; }
    if constexpr (VEC == 2) { v[0] = t.x; v[1] = t.y; }
    if constexpr (VEC == 4) { v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w; }
}

template <int VEC>
__device__ __forceinline__ void store_vec(float *p, const float (&v)[VEC])
{
    using T = typename VecT<VEC>::type;
    T t;
    if constexpr (VEC == 1) { t = v[0]; }
    if constexpr (VEC == 2) { t.x = v[0]; t.y = v[1]; }
    if constexpr (VEC == 4) { t.x = v[0]; t.y = v[1]; t.z = v[2]; t.w = v[3]; }
    *reinterpret_cast<T *>(p) = t;
}

struct TileMap {
    uint32_t ntiles;      // column tiles
    uint32_t nrowgroups;  // groups of kWavesPerGroup rows
    uint32_t mode;        // 0 plain, 1: ntiles divides 8, 2: 8 divides ntiles
};

// Workgroup id -> (column tile, row group).  XCD = id % 8.
__device__ __forceinline__ bool map_tile(const TileMap tm, uint32_t wg, uint32_t &tile, uint32_t &rg)
{
    const uint32_t xcd = wg & 7u, q = wg >> 3;
    if (tm.mode == 1) {
        const uint32_t per = 8u / tm.ntiles;  // XCDs sharing one tile
        tile = xcd % tm.ntiles;
        rg = xcd / tm.ntiles + per * q;
    } else if (tm.mode == 2) {
        const uint32_t per = tm.ntiles >> 3;  // tiles per XCD
        tile = xcd + 8u * (q % per);
        rg = q / per;
    } else {
        tile = wg % tm.ntiles;
        rg = wg / tm.ntiles;
    }
    return rg < tm.nrowgroups;
}

// FULL: every column tile is complete (C % (64*VEC) == 0), no lane predicate.
// kUnroll: gathers per register batch (two batches are in flight).  8 when the
// chip is full of waves; 32 for launches with only a few waves, where a wave's own
// memory latency is all there is to hide.
template <int VEC, int ACT, bool FULL, int kUnroll>
__global__ __launch_bounds__(kWavesPerGroup * 64)
void ellpack_matmul_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx,
                           const uint32_t *__restrict__ nnz, uint32_t m, uint32_t r,
                           const float *__restrict__ X, uint32_t C,
                           const float *__restrict__ bias, float *__restrict__ Y, TileMap tm)
{
    uint32_t tile, rg;
    if (!map_tile(tm, blockIdx.x, tile, rg)) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t row = __builtin_amdgcn_readfirstlane(rg * kWavesPerGroup + (threadIdx.x >> 6));
    if (row >= m) return;

    const uint32_t col = tile * (64u * VEC) + lane * VEC;
    // A partial tile only happens with VEC == 1 (the host picks VEC so that C % VEC == 0).
    const bool live = FULL || col < C;
    const uint32_t cnt = nnz[row];
    const float *__restrict__ wrow = Wd + (size_t)row * r;
    const uint32_t *__restrict__ irow = idx + (size_t)row * r;
    const float *__restrict__ xcol = X + (live ? col : 0u);

    float acc[VEC];
    const float b = bias ? bias[row] : 0.0f;
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = b;

    // Batches of kUnroll nonzeros, double-buffered in registers: the gathers of
    // batch b+1 are issued before batch b is consumed, so a wave always has one
    // batch of loads in flight while it waits for scalar loads or does FMAs.
    // The FMAs themselves stay strictly in slot order.
    float wa[kUnroll], wb[kUnroll];
    float xa[kUnroll][VEC], xb[kUnroll][VEC];
    auto issue = [&](uint32_t j0, float (&w)[kUnroll], float (&x)[kUnroll][VEC]) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            w[u] = wrow[j0 + u];
            load_vec<VEC>(xcol + (size_t)irow[j0 + u] * C, x[u]);
        }
    };
    auto consume = [&](const float (&w)[kUnroll], const float (&x)[kUnroll][VEC]) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = __builtin_fmaf(w[u], x[u][v], acc[v]);
    };
    const uint32_t nb = cnt / kUnroll;
    if (nb) issue(0, wa, xa);
    uint32_t bi = 0;
    for (; bi + 1 < nb; bi += 2) {
        issue((bi + 1) * kUnroll, wb, xb);
        consume(wa, xa);
        if (bi + 2 < nb) issue((bi + 2) * kUnroll, wa, xa);
        consume(wb, xb);
    }
    if (nb & 1u) consume(wa, xa);
    // The last, partial batch.  With few waves on the chip (kUnroll 32) all its gathers are issued at
    // once (slots past the row's end re-read the row's last nonzero) and the multiply-adds run under
    // a wave-uniform test per slot: one memory round trip instead of one per nonzero.  With the chip
    // full of waves the plain loop is faster (no redundant gathers; other waves hide the latency).
    if constexpr (kUnroll >= 32) {
        if (const uint32_t rem = cnt - nb * kUnroll) {
            const uint32_t j0 = nb * kUnroll;
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const uint32_t j = j0 + min((uint32_t)u, rem - 1u);
                wa[u] = wrow[j];
                load_vec<VEC>(xcol + (size_t)irow[j] * C, xa[u]);
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                if ((uint32_t)u < rem) {
#pragma unroll
                    for (int v = 0; v < VEC; ++v) acc[v] = __builtin_fmaf(wa[u], xa[u][v], acc[v]);
                }
        }
    } else {
        for (uint32_t j = nb * kUnroll; j < cnt; ++j) {
            const float w = wrow[j];
            float x[VEC];
            load_vec<VEC>(xcol + (size_t)irow[j] * C, x);
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = __builtin_fmaf(w, x[v], acc[v]);
        }
    }

    if (live) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = so_epilogue<ACT>(acc[v]);
        store_vec<VEC>(Y + (size_t)row * C + col, acc);
    }
}

template <int VEC, int ACT, int UNROLL = 8>
void launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY)
{
    TileMap tm;
    tm.ntiles = so_ceil_div(C, 64u * VEC);
    tm.nrowgroups = so_ceil_div(E->m, kWavesPerGroup);
    tm.mode = (tm.ntiles <= 8 && 8 % tm.ntiles == 0) ? 1 : (tm.ntiles % 8 == 0 ? 2 : 0);
    uint32_t blocks;
    if (tm.mode == 1) blocks = so_ceil_div(tm.nrowgroups, 8u / tm.ntiles) * 8u;
    else blocks = tm.ntiles * tm.nrowgroups;
    const bool full = C % (64u * VEC) == 0;
    auto k = full ? ellpack_matmul_kernel<VEC, ACT, true, UNROLL> : ellpack_matmul_kernel<VEC, ACT, false, UNROLL>;
    k<<<blocks, kWavesPerGroup * 64, 0, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->m, E->r,
                                                       dX, C, dBias, dY, tm);
}

template <int VEC, int UNROLL = 8>
void launch_act(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias,
                float *dY, int act)
{
    switch (act) {
    case SO_ACT_RELU:    launch<VEC, SO_ACT_RELU, UNROLL>(ctx, E, dX, C, dBias, dY); break;
    case SO_ACT_SIGMOID: launch<VEC, SO_ACT_SIGMOID, UNROLL>(ctx, E, dX, C, dBias, dY); break;
    case SO_ACT_TANH:    launch<VEC, SO_ACT_TANH, UNROLL>(ctx, E, dX, C, dBias, dY); break;
    default:             launch<VEC, SO_ACT_NONE, UNROLL>(ctx, E, dX, C, dBias, dY); break;
    }
}

// ---------------------------------------------------------------------------
// Few rows (a classifier head): rows x column tiles give fewer waves than the chip
// has CUs, so a wave's own gather latency is all there is to hide, and the bytes it
// can keep in flight are bounded by its registers.  Here a workgroup of 16 waves
// shares one (row, 64-column tile): the waves split the row's nonzeros among them
// for the gathers (16 times the loads in flight), park the gathered X segments in
// LDS, and the first wave then runs the multiply-adds over them in slot order
// starting from the bias -- the same rounding sequence as the row kernel.
// ---------------------------------------------------------------------------

constexpr int kShareWaves = 16;
constexpr int kSharePerWave = 32;                           // gathers per wave and chunk
constexpr int kShareChunk = kShareWaves * kSharePerWave;    // slots per chunk: 128 KB of X segments
constexpr size_t kShareLdsBytes = (size_t)kShareChunk * 64 * sizeof(float) + kShareChunk * sizeof(float);

template <int ACT>
__global__ __launch_bounds__(kShareWaves * 64)
void ellpack_matmul_shared_gather_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx,
                                         const uint32_t *__restrict__ nnz, uint32_t r,
                                         const float *__restrict__ X, uint32_t C,
                                         const float *__restrict__ bias, float *__restrict__ Y, uint32_t ntiles)
{
    extern __shared__ __attribute__((aligned(16))) float share_lds[];
    float4 *xs4 = reinterpret_cast<float4 *>(share_lds);   // [kShareChunk / 4][64 lanes][4 slots]
    float *ws = share_lds + (size_t)kShareChunk * 64;      // [kShareChunk]
    const uint32_t tile = blockIdx.x % ntiles, row = blockIdx.x / ntiles;   // the grid is exactly m * ntiles
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = tile * 64u + lane;
    const bool live = col < C;
    const uint32_t cnt = nnz[row];
    const float *__restrict__ wrow = Wd + (size_t)row * r;
    const uint32_t *__restrict__ irow = idx + (size_t)row * r;
    const float *__restrict__ xcol = X + (live ? col : 0u);
    float acc = bias ? bias[row] : 0.0f;

    for (uint32_t s0 = 0; s0 < cnt; s0 += kShareChunk) {
        const uint32_t chunk = min((uint32_t)kShareChunk, cnt - s0);
        const uint32_t w0 = wave * kSharePerWave;        // this wave gathers slots s0 + w0 .. + kSharePerWave
        if (w0 < chunk) {
            const uint32_t mine = min((uint32_t)kSharePerWave, chunk - w0);
            float x[kSharePerWave];
#pragma unroll
            for (int u = 0; u < kSharePerWave; ++u) {    // slots past the wave's share re-read its last one
                const uint32_t j = s0 + w0 + min((uint32_t)u, mine - 1u);
                x[u] = xcol[(size_t)irow[j] * C];
            }
            if (lane < mine) ws[w0 + lane] = wrow[s0 + w0 + lane];
            // four consecutive slots of a lane side by side: the wave that multiplies takes them with one read
#pragma unroll
            for (int u = 0; u < kSharePerWave; u += 4)
                if ((uint32_t)u < mine) xs4[((w0 + u) / 4u) * 64u + lane] = make_float4(x[u], x[u + 1], x[u + 2], x[u + 3]);
        }
        __syncthreads();
        if (wave == 0) {
            // One wave, one instruction at a time: what counts is instructions per slot -- a 16-byte read of four
            // weights (every lane the same address), one of this lane's four operands, four multiply-adds.
            uint32_t s = 0;
            for (; s + 8 <= chunk; s += 8) {
                const float4 wa = *reinterpret_cast<const float4 *>(ws + s), wb = *reinterpret_cast<const float4 *>(ws + s + 4);
                const float4 xa = xs4[(s / 4u) * 64u + lane], xb = xs4[(s / 4u + 1u) * 64u + lane];
                acc = __builtin_fmaf(wa.x, xa.x, acc); acc = __builtin_fmaf(wa.y, xa.y, acc);
                acc = __builtin_fmaf(wa.z, xa.z, acc); acc = __builtin_fmaf(wa.w, xa.w, acc);
                acc = __builtin_fmaf(wb.x, xb.x, acc); acc = __builtin_fmaf(wb.y, xb.y, acc);
                acc = __builtin_fmaf(wb.z, xb.z, acc); acc = __builtin_fmaf(wb.w, xb.w, acc);
            }
            for (; s < chunk; ++s) acc = __builtin_fmaf(ws[s], share_lds[(s / 4u) * 256u + lane * 4u + (s & 3u)], acc);
        }
        __syncthreads();                                  // the next chunk overwrites what wave 0 was reading
    }
    if (wave == 0 && live) Y[(size_t)row * C + col] = so_epilogue<ACT>(acc);
}

template <int ACT>
so_status launch_shared_gather(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY)
{
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_matmul_shared_gather_kernel<ACT>));
    const uint32_t ntiles = so_ceil_div(C, 64u);
    ellpack_matmul_shared_gather_kernel<ACT><<<E->m * ntiles, kShareWaves * 64, kShareLdsBytes, ctx->stream>>>(
        E->d_Wd, E->d_idx, E->d_nnz, E->r, dX, C, dBias, dY, ntiles);
    return SO_OK;
}

} // namespace

namespace {

// The row kernel, or the shared-gather one, where X is at most as large as LDS.  The longer of two: the longest row's chain, and two thirds of the mean ones
// that share its SIMD; or the gathers of all nonzeros and the rows' own lines of memory, which long padding spreads; and with many rows the longest one
// may begin late.  Us; fitted as so_matmul_columns_estimate, and as close.
double rows_estimate_small_x(const so_ctx *ctx, const so_ellpack *E)
{
    const double m = E->m, longest = E->max_nnz, mean = (double)E->total_nnz / m, per_simd = std::min(8.0, m / (4.0 * ctx->compute_units));
    if (m <= ctx->compute_units && longest >= 128) return 3.0 + 0.0135 * longest;
    const double chain = longest + 0.63 * mean * std::max(0.0, per_simd - 1.0), lines = m * (1.0 + 0.85 * std::min(1.0, longest / 256.0));
    return 0.4 + std::max(2.05 + 0.0201 * chain, 1.054e-5 * (double)E->total_nnz + 1.68e-4 * lines) + 0.0153 * longest * std::min(1.0, m / 20000.0);
}

// The kernel with X in LDS (csrc/matmul_columns.hip) in place of the row and shared-gather kernels, whose bits it gives: where it applies,
// the longest row has kColumnsNnz nonzeros and it is estimated the faster.  Of 473 launches of up to 400 000 rows, even, skewed or all short
// but one, the choice was the slower one by more than 5 % in 30, by 13 % on average; the longest row alone chose wrongly in 96, by 22 %.
// Us, row or shared-gather kernel / this one, one handle launched again and again, rows x columns x dense columns:
//
//   even rows of    512    1000 x 512 x 32   11.4 /  8.1    1000 x 512 x 1     11.7 /  7.5
//                   383    1337 x 2085 x 1   14.5 /  6.8
//                  2031    489 x 4566 x 4    41.7 / 24.8
//                  1147    12 x 5634 x 1     19.6 / 14.5
//                  1500    17843 x 7108 x 4   293 / 79
//                   112    315 x 140 x 34     4.7 /  3.9
//                   150    4096 x 600 x 64    9.8 /  7.4      60   50 000 x 600 x 64   42.6 / 52.3  (a workgroup copies 154 KB)
//   short, one long        50 000 x 600 x 64 rows of 8 and one of 64   20.8 / 34.7     200 000, of 5 and one of 48   55.4 / 138
//   below kColumnsNnz      1357 x 26 x 8, 20  3.5 /  3.9    2120 x 254 x 3, 42  4.2 / 3.9; faster where there are many rows
constexpr uint32_t kColumnsNnz = 48;

bool columns_pays(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    if (ctx->tune.matmul_columns >= 0) return ctx->tune.matmul_columns == 1 && so_matmul_columns_applies(ctx, E, C);
    // (an override that asks for one of the row kernels' forms stands)
    return ctx->tune.matmul_share < 0 && ctx->tune.matmul_vec == 0 && E->max_nnz >= kColumnsNnz && so_matmul_columns_applies(ctx, E, C) &&
           so_matmul_columns_estimate(ctx, E, C) < rows_estimate_small_x(ctx, E);
}

enum class RbmKernel { None, Merged, Quad, Vector, Planes, Narrow, Slabs };

// Which of the kernels for handles with the RBM layout a launch takes, or None for the kernels below, by estimated
// time.  Both sides of each line were measured, us with one handle launched again and again, in brackets with 48 handles
// and X in turn, whose weights come from memory:
//   quad against the row kernel: 2048 x 2048 x 64 at 95 / 90 / 80 / 50 % sparse 8.1 / 8.8 / 10.1 / 11.7 [8.6 / 9.8 / 11.3 / 13.5]
//   against 6.6 / 9.9 / 16.9 / 35.6 [9.2 / 15.5 / 39.9 / 85.4]; 1024 x 1024 x 64 at 90 / 70 / 50 % 7.0 / 7.5 / 7.8 [7.3 / 7.8 / 8.1]
//   against 5.1 / 9.1 / 13.0 [7.1 / 14.2 / 25.7] -- the row kernel moves 256 bytes per nonzero and 64 columns at about
//   11 TB/s (half of that with the weights from memory), and a row takes 18 ns per nonzero on its own;
//   quad against row-block-merged: 4096 x 4096 x 256 at 90 / 80 / 70 / 50 % 45 / 60 / 72 / 91 against 29 / 48 / 65 / 97
//   -- 2.85 us per million (nonzero, 64 columns) on top of 9.5, and no faster on fewer workgroups than compute units.
//   One to three columns: so_matvec's row kernel on each, which spreads a row over the lanes, from rows of 64 nonzeros
//   per column.  The row kernel has C lanes at work and fetches a line of X per nonzero.  Longest row, us row kernel /
//   that one: one column, 4096 x 4096 1756 101.8 / 9.1, 479 19.7 / 4.8, 159 7.9 / 4.1, 69 4.6 / 4.0; 1024 x 4096
//   62 3.7 / 3.7; 4096 x 512 23 3.5 / 3.9; 10 x 512 63 4.0 / 3.2, 16 3.2 / 3.4; two, 4096 x 4096 487 19.6 / 8.4, 162
//   7.8 / 7.4; 10 x 512 262 6.0 / 3.4; three, 4096 x 4096 1759 114 / 27, 487 19.7 / 13.1; 4096 x 1024 244 11.0 / 10.4.
// `plan` is set where it is Quad: the search for it is the larger part of this function's 0.2 (two K tiles) to 0.6 us (16).
// `us`: the estimate.
RbmKernel rbm_kernel_but_planes(const so_ctx *ctx, const so_ellpack *E, uint32_t C, so_quad_plan *plan, double *us)
{
    const bool merged = so_matmul_rbm_applies(ctx, E, C), quad = so_matmul_quad_applies(ctx, E, C);
    // Below `limit`?  A recording cannot grow the workspace: the quad kernel is then for what has been reserved (the others
    // but the row-block-merged one, which refuses, need none).
    const auto quad_below = [&](double limit) {
        if (!quad || ctx->tune.matmul_quad == 0 || limit <= kQuadLeastUs) return false;
        *plan = so_matmul_quad_choose(ctx, E, C);
        return plan->us < limit && (!ctx->capturing || so_matmul_quad_ready(ctx, *plan));
    };
    if (ctx->tune.matmul_quad == 1 && quad_below(1e30)) { *us = 0.0; return RbmKernel::Quad; }
    const double cus = ctx->compute_units, slabs = so_ceil_div(C, 64), work = (double)E->total_nnz * slabs;
    const bool shared = (double)E->m * slabs <= cus && E->max_nnz >= 128;      // the shared-gather kernel
    *us = 2.5 + std::max(work * 256.0 / 11e6, (shared ? 0.0135 : 0.018) * E->max_nnz + 0.5);
    if (columns_pays(ctx, E, C)) *us = so_matmul_columns_estimate(ctx, E, C);      // which is then what runs in their place
    RbmKernel k = RbmKernel::None;
    if (merged) {
        // one workgroup per (128 rows, 64 columns, share of the columns): pays when that grid covers most of the chip
        const double wgs = (double)E->rbmm.nb * slabs * E->rbmm.ksplit;
        const double t = 9.5 + 2.85e-6 * work * std::ceil(wgs / cus) * cus / wgs;
        if (4.0 * wgs >= 3.0 * cus && (t < *us || !quad)) { *us = t; k = RbmKernel::Merged; }
    }
    if (!quad_below(0.95 * *us)) return k;
    *us = plan->us;
    return RbmKernel::Quad;
}

// The bf16-planes kernel where it is estimated a tenth below the others: us, planes against the fastest of them, one handle launched
// again and again: 4096 x 4096 x 256 at 50 / 70 / 80 % sparse 45 / 44 / 43 against 84 (quad) / 61 / 43 (merged); 3001 x 2777 x 101 at
// 70 % 18.5 against 27.1 (merged); 2048 x 2048 x 256 at 60 / 80 % 17.0 / 16.9 against 23.4 / 18.1 (quad); 4096 x 1024 x 200 at 70 %
// 15.8 against 19.6; 1024 x 4096 x 200 at 70 % 18.4 against 22.2; 2048 x 2048 x 128 at 70 % 14.8 against 14.1; 4096 x 784 x 256 at 90 % 15.0 against 10.8.
constexpr double kPlanesBelow = 0.9;

// The narrow kernel where it is estimated a little below the others.  Of 241 drawn launches (10..4096 rows, 512..4096 columns, 4..256 dense ones, 14 of up to
// 40 000 rows) it is then in no case the slower one by more than 1 %; in nine, the others' choice is slower by 3 to 9 %.  Us, the others and the narrow one, one handle launched again
// and again: column kernel 2847 x 1952 x 8 at 61 % sparse 11.5 / 5.9, 4096 x 2048 x 16 at 50 % 15.2 / 9.3, 20 000 x 600 x 32 at 90 % 9.5 / 14.0; quad 139 x 1436 x 4 at 60 %
// 7.2 / 3.7, 2048 x 2048 x 64 at 80 % 9.9 / 9.6, 2000 x 1500 x 64 at 60 % 9.9 / 11.6, 20 000 x 600 x 64 at 90 % 17.6 / 25.3; row 107 x 730 x 16 at 94 % 3.6 / 3.9.
// In place of so_matvec's row kernel at two and three columns from a million nonzeros on: 1.39 million, two columns, 8.8 / 4.0; 1.5 million, three, 9.6 / 4.3; 2.9 million,
// three, 17.7 / 6.3.  (Below it would gain less, 0.3 to 0.6 of 4.1; with one column it is not looked at.)
//
// At 17 to 32 columns (one slab of 32) its launches of less than 6 us take 0.3 to 0.8 more than estimated, of X with fewer rows than what that was fitted on most; the others'
// less.  Us, columns or row kernel / narrow: 979 x 223 x 19 at 57 % sparse 3.6 / 4.3, 7064 x 109 x 31 at 70 % 4.6 / 5.4, 123 x 168 x 23 at 54 % 3.4 / 3.9; beyond, 8815 x 295 x 29 at 48 % 10.0 / 7.6.  Of
// 543 drawn launches of 16..4000 columns that it took without this term it was 0.4 % the slower one on average, in 203 by more than 4 %; with it, 2.6 % the faster one, in 8 slower by that.
constexpr double kNarrowBelow = 0.955, kNarrowWide = 0.7, kNarrowWideBelow = 6.0;
constexpr uint64_t kNarrowVectorNnz = 1000000;

// The same with X in LDS a part at a time, where it is estimated 7 % below what would run: of 200 drawn launches it is then taken in 47, all of
// them faster, by 17 % on average.  Us, the others and this one: quad 12 x 1238 x 173 at 55 % sparse 7.2 / 5.0, 2000 x 2600 x 16 at 60 % 12.9 / 9.0, 30 x 2988 x 56 at 54 % 7.3 / 7.6,
// 2000 x 1500 x 64 at 60 % 9.9 / 10.5; shared-gather 26 x 745 x 91 at 69 % 5.9 / 4.9, 10 x 1391 x 138 at 82 % 6.0 / 6.2; narrow 17 x 1090 x 28 at 67 % 6.0 / 4.7, 2000 x 1500 x 8 at 60 % 4.6 / 6.8.
constexpr double kSlabsBelow = 0.93;

RbmKernel rbm_kernel(const so_ctx *ctx, const so_ellpack *E, uint32_t C, so_quad_plan *plan, so_planes_plan *planes, so_narrow_plan *narrow)
{
    if (ctx->tune.matmul_rbm == 1 && so_matmul_rbm_applies(ctx, E, C)) return RbmKernel::Merged;
    if (ctx->tune.matmul_rbm == 0) return RbmKernel::None;
    if (ctx->tune.matmul_narrow == 1 && so_matmul_narrow_applies(ctx, E, C)) {
        *narrow = so_matmul_narrow_choose(ctx, E, C);
        return RbmKernel::Narrow;
    }
    if (ctx->tune.matmul_slabs > 0 && so_matmul_slabs_applies(ctx, E, C)) {
        *narrow = so_matmul_slabs_choose(ctx, E, C);
        return RbmKernel::Slabs;
    }
    const bool have = ctx->tune.matmul_planes != 0 && so_matmul_planes_applies(ctx, E, C);
    const bool vector = C <= 3 && E->max_nnz >= 64u * C;
    double us = 0.0;
    RbmKernel k = RbmKernel::Vector;
    if (!vector || (have && ctx->tune.matmul_planes == 1)) k = rbm_kernel_but_planes(ctx, E, C, plan, &us);
    if (have && (!vector || ctx->tune.matmul_planes == 1)) {
        *planes = so_matmul_planes_choose(ctx, E->m, E->n, C);
        if ((ctx->tune.matmul_planes == 1 || planes->us < kPlanesBelow * us) && (!ctx->capturing || so_matmul_planes_ready(ctx, *planes))) {
            k = RbmKernel::Planes;
            us = planes->us;
        }
    }
    // (an override that forces another kernel, or forbids the quad-union copy's, stands)
    if (ctx->tune.matmul_quad >= 0 || ctx->tune.matmul_planes == 1) return k;
    if (ctx->tune.matmul_narrow != 0 && so_matmul_narrow_applies(ctx, E, C)) {
        *narrow = so_matmul_narrow_choose(ctx, E, C);
        const double below = kNarrowBelow * us, wide = narrow->groups == 8u && narrow->slabs == 1u && narrow->us < kNarrowWideBelow ? kNarrowWide : 0.0;
        if (narrow->us < below) us = narrow->us;                          // (what X in parts is compared with)
        if (vector ? C >= 2 && E->total_nnz >= kNarrowVectorNnz : narrow->us + wide < below) k = RbmKernel::Narrow;
    }
    if (vector || ctx->tune.matmul_slabs == 0 || !so_matmul_slabs_applies(ctx, E, C)) return k;
    const so_narrow_plan slabs = so_matmul_slabs_choose(ctx, E, C);
    if (slabs.us >= kSlabsBelow * us) return k;
    // What a recording takes does not change with this kernel, which needs no workspace: the copy's kernels with a reservation, the reference's order without.
    if (ctx->capturing && k != RbmKernel::Narrow && !(so_matmul_quad_applies(ctx, E, C) && so_matmul_quad_ready(ctx, so_matmul_quad_choose(ctx, E, C)))) return k;
    *narrow = slabs;
    return RbmKernel::Slabs;
}

} // namespace

// Widths from one slab to the widest of the fully connected layers this was measured on.
bool so_planes_pays(const so_ctx *ctx, const so_ellpack *E)
{
    if (ctx->tune.matmul_planes >= 0) return ctx->tune.matmul_planes == 1;
    for (uint32_t C : {64u, 128u, 256u}) {
        so_quad_plan plan;
        double us;
        (void)rbm_kernel_but_planes(ctx, E, C, &plan, &us);
        if (so_matmul_planes_choose(ctx, E->m, E->n, C).us < kPlanesBelow * us) return true;
    }
    return false;
}

extern "C" so_status so_matmul_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    SO_REQUIRE(ctx && E, "so_matmul_reserve: null argument");
    if (E->m == 0 || C == 0) return SO_OK;
    // All kernels of the layout: which one runs is settled at launch, where the tuning overrides may have changed.
    so_status st = SO_OK;
    if (so_matmul_quad_applies(ctx, E, C)) st = so_matmul_quad_reserve(ctx, E, C);
    if (st == SO_OK && so_matmul_planes_applies(ctx, E, C)) st = so_matmul_planes_reserve(ctx, E, C);
    if (st == SO_OK && so_matmul_rbm_applies(ctx, E, C)) {
        st = so_matmul_rbm_reserve(ctx, E, C);
        if (st == SO_OK) st = so_matmul_rbm_set_pitch(ctx, E, C);
    }
    return st;
}

extern "C" so_status so_matmul(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C,
                               const float *dBias, float *dY, int act)
{
    SO_REQUIRE(ctx && E, "so_matmul: null argument");
    SO_REQUIRE(act >= SO_ACT_NONE && act <= SO_ACT_TANH, "so_matmul: unknown activation %d", act);
    if (E->m == 0 || C == 0) return SO_OK;  // empty output: nothing to launch
    SO_REQUIRE(dY != nullptr, "so_matmul: Y is null");
    SO_REQUIRE(dX != nullptr || E->total_nnz == 0, "so_matmul: X is null");
    // one workgroup per (4 rows, 64 columns) at most: the grid must fit 31 bits
    SO_REQUIRE(((uint64_t)E->m / 4 + 8) * ((uint64_t)C / 64 + 1) < (1ull << 31), "so_matmul: %u x %u output is too large for one launch", E->m, C);

    // The kernels of the RBM layout, on handles uploaded with it (accurate to fp32 round-off, not bit-identical to
    // the row order: the caller asked for them by asking for the layout; SPARSEOPS_MATMUL_RBM=0 forbids all of them, =1
    // forces the row-block-merged one, SPARSEOPS_MATMUL_QUAD=1 / 0 forces / forbids the quad-union one, SPARSEOPS_MATMUL_PLANES the bf16-planes one, SPARSEOPS_MATMUL_NARROW the narrow one, SPARSEOPS_MATMUL_SLABS the one with X a part at a time).
    if ((E->layouts & SO_LAYOUT_RBM) && dX != nullptr && (((uintptr_t)dX | (uintptr_t)dY) & 3) == 0) {
        so_quad_plan plan;
        so_planes_plan pplan;
        so_narrow_plan nplan;
        const RbmKernel k = rbm_kernel(ctx, E, C, &plan, &pplan, &nplan);
        if (k != RbmKernel::None) {
            const so_status st = k == RbmKernel::Quad ? so_matmul_quad_launch(ctx, E, plan, dX, C, dBias, dY, act)
                               : k == RbmKernel::Narrow || k == RbmKernel::Slabs ? so_matmul_narrow_launch(ctx, E, nplan, dX, C, dBias, dY, act)
                               : k == RbmKernel::Planes ? so_matmul_planes_launch(ctx, E, pplan, dX, C, dBias, dY, act)
                               : k == RbmKernel::Vector ? so_matvec_columns(ctx, E, dX, C, dBias, dY, act)
                                                        : so_matmul_rbm_launch(ctx, E, dX, C, dBias, dY, act);
            if (st != SO_OK) return st;
            SO_LAUNCH_CHECK();
            ctx->last_kernel = k == RbmKernel::Quad ? "quad" : k == RbmKernel::Narrow ? "narrow" : k == RbmKernel::Slabs ? "slabs" : k == RbmKernel::Planes ? "planes" : k == RbmKernel::Vector ? "vector" : "merged";
            return SO_OK;
        }
    }

    const uintptr_t align = (uintptr_t)dX | (uintptr_t)dY;
    // The LDS-staged kernel needs whole float4 column groups.  It takes one
    // workgroup per (64 rows, 64 columns), one workgroup per CU at a time, so it pays
    // only when that grid covers most of the chip; smaller problems stay on the row
    // kernel (SPARSEOPS_MATMUL_TILED=1 forces it, =0 forbids it: tuning and tests).
    bool tiled = (E->layouts & SO_LAYOUT_TILED) && C % 4 == 0 && C >= 16 && (align & 15) == 0 &&
                 (size_t)ctx->max_lds_bytes >= so_tiled::kLdsBytes;
    if (tiled) {
        const uint64_t groups = (uint64_t)so_ceil_div(C, so_tiled::kSlabCols) * so_ceil_div(E->tiled.nquads, so_tiled::kWavesPerGroup);
        if (ctx->tune.matmul_tiled >= 0) tiled = ctx->tune.matmul_tiled == 1;
        else tiled = 4 * groups >= 3 * (uint64_t)ctx->compute_units;
    }
    if (tiled) {
        const so_status st = so_matmul_tiled_launch(ctx, E, dX, C, dBias, dY, act);
        if (st != SO_OK) return st;
        SO_LAUNCH_CHECK();
        ctx->last_kernel = "tiled";
        return SO_OK;
    }

    if (dX != nullptr && (((uintptr_t)dX | (uintptr_t)dY) & 3) == 0 && columns_pays(ctx, E, C)) {
        const so_status st = so_matmul_columns_launch(ctx, E, dX, C, dBias, dY, act);
        if (st != SO_OK) return st;
        SO_LAUNCH_CHECK();
        ctx->last_kernel = "columns";
        return SO_OK;
    }

    // Columns per lane: as wide as alignment allows while every tile stays whole.
    int vec = 1;
    if (C % 256 == 0 && (align & 15) == 0) vec = 4;
    else if (C % 128 == 0 && (align & 7) == 0) vec = 2;
    if ((ctx->tune.matmul_vec == 1 || ctx->tune.matmul_vec == 2) && ctx->tune.matmul_vec < vec) vec = ctx->tune.matmul_vec;   // narrower lanes only
    // Few waves in total (at most one per SIMD even with one column per lane): the
    // launch is latency-bound, so spread it over as many waves as possible and give
    // each wave 2 x 32 gathers in flight.
    const uint64_t row_tiles = (uint64_t)E->m * so_ceil_div(C, 64);
    // At most one (row, tile) per CU and rows long enough to be worth sharing: 16 waves gather for each.
    bool share = row_tiles <= (uint64_t)ctx->compute_units && E->max_nnz >= 128 && (size_t)ctx->max_lds_bytes >= kShareLdsBytes;
    if (ctx->tune.matmul_share >= 0) share = share && ctx->tune.matmul_share == 1;
    if (share) {
        so_status st;
        switch (act) {
        case SO_ACT_RELU:    st = launch_shared_gather<SO_ACT_RELU>(ctx, E, dX, C, dBias, dY); break;
        case SO_ACT_SIGMOID: st = launch_shared_gather<SO_ACT_SIGMOID>(ctx, E, dX, C, dBias, dY); break;
        case SO_ACT_TANH:    st = launch_shared_gather<SO_ACT_TANH>(ctx, E, dX, C, dBias, dY); break;
        default:             st = launch_shared_gather<SO_ACT_NONE>(ctx, E, dX, C, dBias, dY); break;
        }
        if (st != SO_OK) return st;
        SO_LAUNCH_CHECK();
        ctx->last_kernel = "shared";
        return SO_OK;
    }
    if (row_tiles <= 4ull * (uint64_t)ctx->compute_units && E->max_nnz >= 64)
        launch_act<1, 32>(ctx, E, dX, C, dBias, dY, act);
    else if (vec == 4) launch_act<4>(ctx, E, dX, C, dBias, dY, act);
    else if (vec == 2) launch_act<2>(ctx, E, dX, C, dBias, dY, act);
    else launch_act<1>(ctx, E, dX, C, dBias, dY, act);
    SO_LAUNCH_CHECK();
    ctx->last_kernel = "row";
    return SO_OK;
}
