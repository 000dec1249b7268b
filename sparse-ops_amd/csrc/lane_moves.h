// Values moved between the lanes of a wave inside the vector unit: DPP controls within a row of 16 lanes, v_permlane16_swap and v_permlane32_swap
// across rows.  An exchange through LDS (what __shfl_xor compiles to) takes some 100 clocks, and a reduction is six of them one after the other: 0.25 us of a
// matvec's 4, 0.2 to 0.3 of the encoder's 16.4 on 400 x 700.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace so_lanes {

template <int CONTROL, int BANKS = 0xf>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CONTROL, 0xf, BANKS, false);
}

// The word of the lane `D` away (lane number ^ D), D = 8, 4, 2 or 1: a rotation of the row, the two halves of a shift, or a permutation of four lanes.
template <int D>
__device__ __forceinline__ uint32_t word_across(uint32_t v)
{
    static_assert(D == 8 || D == 4 || D == 2 || D == 1, "within a row of 16");
    if constexpr (D == 8) return dpp<0x128>(v, v);                                   // row_ror:8
    else if constexpr (D == 4) return dpp<0x114, 0xa>(dpp<0x104, 0x5>(v, v), v);     // row_shl:4 for the even fours, row_shr:4 for the odd
    else if constexpr (D == 2) return dpp<0x4e>(v, v);                               // quad_perm: [2, 3, 0, 1]
    else return dpp<0xb1>(v, v);                                                     // [1, 0, 3, 2]
}

template <int D>
__device__ __forceinline__ float across(float v) { return __uint_as_float(word_across<D>(__float_as_uint(v))); }

// op over a value of G lanes (64, 32, 16, 8 or 4, aligned), in all of them: pairs G / 2 apart first, then G / 4 and so on; op is commutative.  All G lanes
// are active.  4- and 8-byte values.
template <int G, class T, class Op>
__device__ __forceinline__ T reduce(T v, Op op)
{
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one word or two");
    constexpr int words = sizeof(T) / 4;
    struct Words { uint32_t w[words]; };
    const auto step = [&](auto move) {                                               // move(word, first, second): the two that meet
        const Words a = __builtin_bit_cast(Words, v);
        Words p, q;
#pragma unroll
        for (int i = 0; i < words; ++i) move(a.w[i], p.w[i], q.w[i]);
        v = op(__builtin_bit_cast(T, p), __builtin_bit_cast(T, q));
    };
    if constexpr (G >= 64)
        step([](uint32_t w, uint32_t &p, uint32_t &q) { const auto h = __builtin_amdgcn_permlane32_swap(w, w, false, false); p = h[0]; q = h[1]; });
    if constexpr (G >= 32)
        step([](uint32_t w, uint32_t &p, uint32_t &q) { const auto h = __builtin_amdgcn_permlane16_swap(w, w, false, false); p = h[0]; q = h[1]; });
    if constexpr (G >= 16) {
        step([](uint32_t w, uint32_t &p, uint32_t &q) { p = w; q = word_across<8>(w); });
        step([](uint32_t w, uint32_t &p, uint32_t &q) { p = w; q = dpp<0x124>(w, w); });      // row_ror:4: the halves of a row are the same by now
    } else if constexpr (G == 8) {
        step([](uint32_t w, uint32_t &p, uint32_t &q) { p = w; q = word_across<4>(w); });
    }
    step([](uint32_t w, uint32_t &p, uint32_t &q) { p = w; q = word_across<2>(w); });
    step([](uint32_t w, uint32_t &p, uint32_t &q) { p = w; q = word_across<1>(w); });
    return v;
}

struct Sum { template <class T> __device__ __forceinline__ T operator()(T a, T b) const { return a + b; } };
struct Max { __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return max(a, b); } };

} // namespace so_lanes
