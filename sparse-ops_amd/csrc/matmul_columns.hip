// so_matmul for few rows and at most 64 dense columns, in the row kernels' order: a classifier head, the small layers of a model.
//
// A launch with at most a few waves per SIMD is as long as its longest row's chain.  The row kernel gathers from memory and pays some
// 43 clocks an entry; here all of X lies in LDS (n * C values) and a lane is one dense column, as in the column convolution
// (csrc/conv_columns.hip): an entry is an address add, a 4-byte LDS read and a multiply-add, the row's (weight, X row) pairs held
// 16 at a time in lanes and handed round by DPP, reads three quads of entries ahead.  With at most 16 or 32 columns a wave
// takes four or two rows, 16 or 32 lanes each.  Bias first, then one multiply-add per stored nonzero in slot order: same bits as
// the row kernels.
//
// What bounds it: about 20 clocks an entry of the longest row on a SIMD of its own (what one wave alone issues), after 3.5 us of launch and the
// copy of X; with many rows the copies, one of all of X per workgroup.
#include "so_internal.h"
#include "dpp_steps.h"
#include "lds_sync.h"

#include <algorithm>
#include <cmath>

namespace {

using so_dpp::fma4;
using so_dpp::step4;

// RPW rows per wave, 64 / RPW lanes each.
template <int RPW, int ACT>
__global__ __launch_bounds__(1024)
void ellpack_matmul_columns_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx, const uint32_t *__restrict__ nnz, uint32_t m, uint32_t r,
                                   const float *__restrict__ X, uint32_t n, uint32_t C, const float *__restrict__ bias, float *__restrict__ Y)
{
    extern __shared__ __attribute__((aligned(16))) float xs[];         // X, then a row of zeros for the padding entries
    constexpr uint32_t LPR = 64u / RPW;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, threads = blockDim.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t row = (blockIdx.x * (threads / 64u) + wave) * RPW + lane / LPR, col = lane % LPR;
    const uint32_t safe = min(row, m - 1u), have = nnz[safe], cnt = row < m ? have : 0u;
    const float *__restrict__ wr = Wd + (size_t)safe * r;
    const uint32_t *__restrict__ ir = idx + (size_t)safe * r;
    const uint32_t l16 = lane & 15u, pitch = C * 4u, pad = n * pitch, last = max(cnt, 1u) - 1u;
    uint32_t longest = cnt;
#pragma unroll
    for (uint32_t off = LPR; off < 64u; off <<= 1) longest = max(longest, (uint32_t)__shfl_xor(longest, off, 64));
    const uint32_t groups = __builtin_amdgcn_readfirstlane((longest + 15u) / 16u);

    // a group of 16 entries: weight and LDS offset, in the lanes of each row of 16
    float w[4], wn[4];
    uint32_t o[4], on[4];
    auto ask = [&](uint32_t g, float &we, uint32_t &oe) {
        const uint32_t k = min(g * 16u + l16, last);
        we = wr[k];
        oe = ir[k];
    };
    auto settle = [&](uint32_t g, float &we, uint32_t &oe) {
        const bool in = g * 16u + l16 < cnt;
        we = in ? we : -0.0f;
        oe = in ? oe * pitch : pad;
    };
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) ask(i, w[i], o[i]);
    float acc = bias ? bias[safe] : 0.0f;

    // X straight from memory into LDS, 16 bytes per lane; what is left, by the word
    const uint32_t values = n * C, quads = values / 4u;
    const uint32_t lds0 = so_lds::lds_address(xs) + wave * 1024u;
    if ((reinterpret_cast<uintptr_t>(X) & 15u) == 0u) {
        uint32_t to = lds0;
        for (uint32_t q = tid; q < quads; q += threads, to += threads * 16u)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(__builtin_amdgcn_readfirstlane(to)), "v"(q * 16u), "s"(X) : "memory", "m0");
        for (uint32_t k = quads * 4u + tid; k < values; k += threads) xs[k] = X[k];
    } else {
        for (uint32_t k = tid; k < values; k += threads) xs[k] = X[k];
    }
    if (tid < C) xs[values + tid] = 0.0f;
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");                 // this thread's part of X is in LDS
    __syncthreads();

    const uint32_t base = so_lds::lds_address(xs) + (col < C ? col * 4u : 0u);
    float xA[4], xB[4] = {0.f, 0.f, 0.f, 0.f}, xC[4] = {0.f, 0.f, 0.f, 0.f}, xD[4] = {0.f, 0.f, 0.f, 0.f}, owed = -0.0f;
    auto group = [&](float we, uint32_t off) {
        asm volatile("s_nop 4" : "+v"(we), "+v"(off), "+v"(owed));      // DPP operands: not within two cycles of a vector write
        step4<0, 4>(base, off, xA, owed, xB, acc);
        step4<4, 8>(base, off, xB, owed, xC, acc);
        step4<8, 12>(base, off, xC, owed, xD, acc);
        step4<12, 0>(base, off, xD, we, xA, acc);
        owed = we;
    };
    for (uint32_t g = 0; g < groups; g += 4u) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) ask(g + 4u + i, wn[i], on[i]);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) settle(g + i, w[i], o[i]);
        group(w[0], o[0]);
        if (g + 1u < groups) group(w[1], o[1]);
        if (g + 2u < groups) group(w[2], o[2]);
        if (g + 3u < groups) group(w[3], o[3]);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) { w[i] = wn[i]; o[i] = on[i]; }
    }
    asm volatile("s_nop 4" : "+v"(owed));
    fma4<4>(owed, xB, acc);
    fma4<8>(owed, xC, acc);
    fma4<12>(owed, xD, acc);
    if (row < m && col < C) Y[(size_t)row * C + col] = so_epilogue<ACT>(acc);
}

size_t columns_lds(const so_ellpack *E, uint32_t C) { return (((size_t)E->n + 1) * C * 4 + 15) / 16 * 16; }

uint32_t rows_per_wave(uint32_t C) { return C <= 16u ? 4u : C <= 32u ? 2u : 1u; }

// Waves of a workgroup: four while that leaves compute units free, else up to 16 that share one copy of X.
uint32_t columns_waves(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    uint32_t waves = 4;
    while (waves < 16 && so_ceil_div(E->m, waves * rows_per_wave(C)) > (uint32_t)ctx->compute_units) waves *= 2;
    return waves;
}

template <int RPW>
so_status launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    const size_t lds = columns_lds(E, C);
    auto k = act == SO_ACT_RELU ? ellpack_matmul_columns_kernel<RPW, SO_ACT_RELU> : act == SO_ACT_SIGMOID ? ellpack_matmul_columns_kernel<RPW, SO_ACT_SIGMOID>
           : act == SO_ACT_TANH ? ellpack_matmul_columns_kernel<RPW, SO_ACT_TANH> : ellpack_matmul_columns_kernel<RPW, SO_ACT_NONE>;
    SO_HIP(so_allow_big_lds(ctx, (const void *)k));
    const uint32_t waves = columns_waves(ctx, E, C);
    k<<<so_ceil_div(E->m, waves * RPW), waves * 64, lds, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->m, E->r, dX, E->n, C, dBias, dY);
    return SO_OK;
}

} // namespace

bool so_matmul_columns_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return C <= 64u && E->total_nnz != 0 && columns_lds(E, C) <= (size_t)ctx->max_lds_bytes;
}

// 1.9 us, then the longer of two: the longest row at 9.9 ns an entry, and as much for the mean ones that share its SIMD; or, as often as the chip is filled
// with workgroups, 1.2 us and 10 ns per KB of X that a compute unit's workgroups copy, and a wave's entries -- its longest row's, which is not known here: at
// most the longest of all, about three or eight times the mean where it takes two or four rows -- at 4.5 ns by wave of a SIMD.  Fitted on 237 launches of 48
// nonzeros and more in the longest row, up to 400 000 rows even, skewed and all short but one; half of 236 others are within 8 %.
double so_matmul_columns_estimate(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    const double cus = ctx->compute_units, kb = (double)columns_lds(E, C) / 1024.0, longest = E->max_nnz, mean = (double)E->total_nnz / E->m;
    const uint32_t rpw = rows_per_wave(C), waves = columns_waves(ctx, E, C);
    const double wgs = so_ceil_div(E->m, waves * rpw);
    const double fit = std::max(1.0, std::min(std::floor((double)ctx->max_lds_bytes / (kb * 1024.0)), std::floor(32.0 / waves)));
    const double filled = std::max(1.0, wgs / (cus * fit)), resident = std::min(fit, wgs / cus);
    const double entries = std::min(longest, mean * (1.0 + 2.4 * (rpw - 1)) + 8.7) * wgs * waves / (4.0 * cus);
    const double chain = longest + mean * std::max(0.0, resident * waves / 4.0 / 1.17 - 1.0);
    return 1.9 + std::max(1.2 + 0.0099 * chain, filled * (1.2 + 0.01 * kb * std::max(1.0, resident)) + 0.0045 * entries);
}

so_status so_matmul_columns_launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    if (C <= 16u) return launch<4>(ctx, E, dX, C, dBias, dY, act);
    if (C <= 32u) return launch<2>(ctx, E, dX, C, dBias, dY, act);
    return launch<1>(ctx, E, dX, C, dBias, dY, act);
}
