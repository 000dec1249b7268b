// Outputs of the quad-union copy's kernels that came out as NaN -- a zero weight of the union met a value of X that is not finite -- from the
// row's own nonzeros.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

typedef float so_f32x4 __attribute__((ext_vector_type(4)));
typedef float so_f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// The outputs of columns col .. col + 3 (col + 3 < a.C; WIDE false: of those that exist, the last one again for the others), added up by the 16 lanes that share the row (lane
// `sub` every 16th, eight of them requested at a time), in an order that depends on the row's length alone.
template <bool WIDE = true, class Args>
__device__ __forceinline__ so_f32x4 exact_outputs(const Args &a, uint32_t row, uint32_t col, uint32_t sub)
{
    constexpr uint32_t AHEAD = 8;
    const uint32_t cnt = row < a.m ? a.nnz[row] : 0u;
    const float *w = a.Wd + (size_t)row * a.r;
    const uint32_t *ix = a.idx + (size_t)row * a.r;
    so_f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t k = sub; k < cnt; k += 16u * AHEAD) {
        float wk[AHEAD];
        so_f32x4 x[AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) {
            const uint32_t at = min(k + 16u * u, cnt - 1u);
            wk[u] = w[at];
            const float *from = a.X + (size_t)ix[at] * a.C + col;
            if constexpr (WIDE) x[u] = *reinterpret_cast<const so_f32x4u *>(from);
            else
#pragma unroll
                for (uint32_t v = 0; v < 4; ++v) x[u][v] = from[min(v, a.C - 1u - col)];
        }
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u)
            if (k + 16u * u < cnt)
#pragma unroll
                for (int v = 0; v < 4; ++v) sum[v] = __builtin_fmaf(wk[u], x[u][v], sum[v]);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1)
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[v] += __shfl_xor(sum[v], off, 64);
    return sum;
}
