// so_matvec: y[m] = E * x[n] + bias on gfx950.
//
// The product is a pure stream of the stored (weight, column) pairs -- 8 bytes
// per nonzero and one multiply-add -- so the kernels are built around HBM
// bandwidth: x is staged once per workgroup in LDS when it fits (the gathers
// then never leave the CU), the pairs are read with 16-byte non-temporal loads,
// four per lane in flight, and only the first nnz[i] slots of a row are touched,
// so ELLPACK padding is never streamed.  A handle uploaded with SO_LAYOUT_IDX16 also has
// its columns in 16 bits: the kernels then stream 6 bytes per nonzero.
//
//   rows kernel    one wavefront per row on the row-major arrays; lanes take
//                  aligned groups of four slots, partial sums are combined with a
//                  butterfly of lane exchanges.
//   binned kernel  one launch over four length classes (skewed matrices): a whole
//                  workgroup for rows of more than 4096 nonzeros, whole waves for
//                  long rows, 16 or 4 lanes per row for short ones; workgroups of
//                  the long classes are dispatched first.
//   slot kernel    one lane per row on the slot-major arrays (consecutive rows'
//                  k-th nonzeros are contiguous, so loads coalesce across lanes).
//
// Reference: ellpack_matvec, src/ellpack_matvec.cpp:20-147.  The reference sums
// 16 interleaved partials and a tree (:72-96); the orders here differ, so results
// agree to fp32 round-off, not bit for bit.
#include "so_internal.h"
#include "lane_moves.h"

#include <algorithm>

namespace {

constexpr int kBlock = 1024;
constexpr int kWavesPerBlock = kBlock / 64;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// The columns of four consecutive slots as they are loaded: four 32-bit words, or two when the
// handle carries its columns in 16 bits as well (SO_LAYOUT_IDX16: 6 bytes per nonzero instead of 8).
template <bool I16> struct ColGroup;
template <> struct ColGroup<false> {
    using T = u32x4;
    using E = uint32_t;
    static __device__ __forceinline__ u32x4 cols(T t) { return t; }
};
template <> struct ColGroup<true> {
    using T = u32x2;
    using E = uint16_t;
    static __device__ __forceinline__ u32x4 cols(T t)
    {
        u32x4 c;
        c.x = t.x & 0xffffu; c.y = t.x >> 16; c.z = t.y & 0xffffu; c.w = t.y >> 16;
        return c;
    }
};

// A launch whose result goes to pinned host memory (TELL): row i is the pair {y[i], turn}, in one store of 8 bytes, so that what the host
// polls is the result itself.  The link takes some 10 ns per store instruction's line, whatever it holds: a workgroup's rows are
// collected in LDS and leave 64 at a time.  (Each row by its own wave: 13 to 40 us more for 1500 to 4096 rows; words of 4 bytes
// with a flag and a fence for all memory per workgroup 20 to 60.)
struct Tell {
    uint2 *rows;
    uint32_t turn;
};

// What a workgroup holds for the host: `per` results of each of its passes, those of pass p from place p * stride + first on.
template <bool TELL>
__device__ __forceinline__ void tell_host(const Tell &tell, const float *held, uint32_t per, uint32_t stride, uint32_t first, uint32_t count, uint32_t at)
{
    if constexpr (TELL) {
        __syncthreads();
        const uint32_t pass = threadIdx.x / per, mine = pass * stride + first + threadIdx.x % per;
        if (mine < count)
            __hip_atomic_store(reinterpret_cast<unsigned long long *>(tell.rows + at + mine), (unsigned long long)tell.turn << 32 | __float_as_uint(held[threadIdx.x]),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The sum over G lanes in all of them, by lane moves (by six exchanges through LDS, one after the other, at the end of a launch: 1000 x 1000 at 70 % sparse
// 4.00 us, so 3.75).
template <int G>
__device__ __forceinline__ float group_sum(float v) { return so_lanes::reduce<G>(v, so_lanes::Sum()); }

// Stage x in LDS (XLDS) or read it through the cache hierarchy.  `pitch`: floats from one element of x to the next.
template <bool XLDS>
__device__ __forceinline__ const float *stage_x(const float *__restrict__ x, uint32_t n, float *lds, uint32_t pitch = 1u)
{
    if (!XLDS) return x;
    if (pitch != 1u) {
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) lds[i] = x[(size_t)i * pitch];
        __syncthreads();
        return lds;
    }
    const uint32_t n4 = ((reinterpret_cast<uintptr_t>(x) & 15u) == 0) ? n / 4 : 0;     // 16-byte copies when x is aligned
    for (uint32_t i = threadIdx.x; i < n4; i += blockDim.x)
        reinterpret_cast<float4 *>(lds)[i] = reinterpret_cast<const float4 *>(x)[i];
    for (uint32_t i = n4 * 4 + threadIdx.x; i < n; i += blockDim.x) lds[i] = x[i];
    __syncthreads();
    return lds;
}

// Dot product of one row with x, computed by a whole wave, in two halves so that a caller can
// put other work (staging x, finishing the previous row) between issuing the loads and using
// them.  The row's slots [beg, end) are covered by aligned groups of four; a lane loads up to four
// such groups (addresses past the row are clamped onto its last group and every slot outside
// [beg, end) is masked to an exact no-op).  Rows longer than 1024 slots continue in row_rest.
template <bool I16>
struct RowLoads {
    f32x4 w[4];
    typename ColGroup<I16>::T c[4];
};

// G = lanes that share a row (64, 32, 16 or 8): a pass of the row covers 16 G slots.
template <int G, bool I16>
__device__ __forceinline__ void row_issue(const f32x4 *__restrict__ Wd4, const typename ColGroup<I16>::T *__restrict__ idx4,
                                          uint64_t beg, uint64_t end, uint64_t q0, RowLoads<I16> &L)
{
    const uint64_t qlast = end > beg ? (end - 1) >> 2 : beg >> 2;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint64_t q = std::min<uint64_t>(q0 + (uint64_t)G * u, qlast);
        L.w[u] = __builtin_nontemporal_load(Wd4 + q);
        L.c[u] = __builtin_nontemporal_load(idx4 + q);
    }
}

// a[j]: the four partial sums of column j of the W dense ones, which lie side by side in xs, `pitch` floats from one element to the next.
// FOURS: the four slots of a group together, which the compiler turns into branches around the last of them: the better code for the row kernel's one column
// (8000 x 8000 at 85 % sparse 12.65 against 13.35 us, 12 000 x 2000 at 95 % 5.98 and 5.88), not for the length classes' waves (Zipf rows, 12 000 x 12 000, 8.57 and 8.43) nor
// for three columns, which spill.
template <int G, bool I16, bool FOURS, int W>
__device__ __forceinline__ void row_consume(const RowLoads<I16> &L, uint64_t beg, uint64_t end, uint64_t q0, const float *xs, float (&a)[W][4], size_t pitch = W)
{
    // slot k of group u is live iff its distance from the row's start is in [0, end - beg): one
    // unsigned 32-bit comparison (a slot before the row gives a huge distance)
    const uint32_t len = (uint32_t)(end - beg);
    const int32_t rel0 = (int32_t)(int64_t)((q0 << 2) - beg);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int32_t rel = rel0 + 4 * G * u;
        const u32x4 c = ColGroup<I16>::cols(L.c[u]);
        if constexpr (FOURS) {
            static_assert(W == 1, "one column");
            const bool v0 = (uint32_t)rel < len, v1 = (uint32_t)(rel + 1) < len;
            const bool v2 = (uint32_t)(rel + 2) < len, v3 = (uint32_t)(rel + 3) < len;
            const float x0 = xs[(v0 ? c.x : 0u) * pitch], x1 = xs[(v1 ? c.y : 0u) * pitch];
            const float x2 = xs[(v2 ? c.z : 0u) * pitch], x3 = xs[(v3 ? c.w : 0u) * pitch];
            a[0][0] = __builtin_fmaf(v0 ? L.w[u].x : 0.0f, v0 ? x0 : 0.0f, a[0][0]);
            a[0][1] = __builtin_fmaf(v1 ? L.w[u].y : 0.0f, v1 ? x1 : 0.0f, a[0][1]);
            a[0][2] = __builtin_fmaf(v2 ? L.w[u].z : 0.0f, v2 ? x2 : 0.0f, a[0][2]);
            a[0][3] = __builtin_fmaf(v3 ? L.w[u].w : 0.0f, v3 ? x3 : 0.0f, a[0][3]);
            continue;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool v = (uint32_t)(rel + k) < len;
            const float *xk = xs + (v ? c[k] : 0u) * pitch;
            const float w = v ? L.w[u][k] : 0.0f;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const float x = xk[j];
                a[j][k] = __builtin_fmaf(w, v ? x : 0.0f, a[j][k]);
            }
        }
    }
}

// The whole row at once (used where rows are not pipelined).
template <bool I16>
__device__ __forceinline__ float wave_row_dot(const f32x4 *__restrict__ Wd4, const typename ColGroup<I16>::T *__restrict__ idx4,
                                              uint64_t beg, uint64_t end, const float *xs, uint32_t lane)
{
    float a[1][4] = {};
    if (end == beg) return 0.0f;
    const uint64_t qlast = (end - 1) >> 2;
    for (uint64_t q0 = (beg >> 2) + lane; q0 <= qlast; q0 += 256) {
        RowLoads<I16> L;
        row_issue<64, I16>(Wd4, idx4, beg, end, q0, L);
        row_consume<64, I16, false>(L, beg, end, q0, xs, a);
    }
    return group_sum<64>((a[0][0] + a[0][1]) + (a[0][2] + a[0][3]));
}

template <int G, typename IdxT>
__device__ __forceinline__ float group_row_dot(const float *__restrict__ Wd, const IdxT *__restrict__ idx,
                                               uint64_t base, uint32_t cnt, const float *xs, uint32_t sub)
{
    float a = 0.0f;
    for (uint32_t j = sub; j < cnt; j += G) a = __builtin_fmaf(Wd[base + j], xs[idx[base + j]], a);
    return group_sum<G>(a);
}

// G lanes per row: a wave works on 64/G rows at a time (whole waves for rows longer than 512
// slots, a half, a quarter or an eighth of a wave for shorter ones, so that short rows do not leave lanes idle).
// MM: so_matmul's products with few columns of row-major X and Y (their rows `C` floats apart), W of them per blockIdx.y, with an activation.
template <bool XLDS, int G, bool I16, int W, bool MM, bool TELL>
__global__ __launch_bounds__(kBlock)
void matvec_rows_kernel(const float *__restrict__ Wd, const void *__restrict__ idx,
                        const uint32_t *__restrict__ nnz, uint32_t count, uint32_t r,
                        const float *__restrict__ x, uint32_t n,
                        const float *__restrict__ bias, float *__restrict__ y, uint32_t C, int act, uint32_t whole, Tell tell)
{
    extern __shared__ float lds_x[];
    static_assert(W == 1 || (MM && XLDS), "several columns at once are all the columns, and in LDS");
    constexpr uint32_t RPW = 64 / G;                                     // rows per wave
    const uint32_t lane = threadIdx.x & 63u, sub = lane % G, grp = lane / G;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6));
    const uint32_t stride = gridDim.x * kWavesPerBlock * RPW;            // rows between a group's consecutive rows
    const f32x4 *Wd4 = reinterpret_cast<const f32x4 *>(Wd);
    const typename ColGroup<I16>::T *idx4 = reinterpret_cast<const typename ColGroup<I16>::T *>(idx);
    // Rows are pipelined: the first 16 G slots of the next row are requested before the current
    // row is reduced, and those of the group's first row before x is staged, so that a wave always
    // has a row's worth of loads in flight.  Row lengths are fetched two rows ahead, so that
    // requesting a row never waits for its length -- nor does the first of a small launch, whose slots are requested up to its pitch (`whole`).
    uint32_t row = wave * RPW + grp, held = threadIdx.x / G;
    const uint64_t first = (uint64_t)row * r;
    RowLoads<I16> cur, nxt;
    const uint32_t len0 = row < count ? nnz[row] : 0u;
    uint32_t len1 = (uint64_t)row + stride < count ? nnz[row + stride] : 0u;          // length of the next row
    uint32_t ask = r;
    if (whole == 0u) {
        ask = len0;
        asm volatile("" : "+v"(ask));                                    // (a branch: a choice of values would wait for the length)
    }
    if (row < count) row_issue<G, I16>(Wd4, idx4, first, first + ask, (first >> 2) + sub, cur);
    uint64_t beg = first, end = beg + len0;
    const uint32_t pitch = MM && W == 1 ? C : 1u;
    const float *xs = stage_x<XLDS>(MM && W == 1 ? x + blockIdx.y : x, n * W, lds_x, pitch);
    const size_t xpitch = XLDS ? W : pitch;
    // all groups of a wave make the same number of trips (the reductions need every lane)
    for (uint32_t base = wave * RPW; base < count; base += stride, row += stride) {
        const uint64_t nrow = (uint64_t)row + stride;
        const uint64_t nbeg = nrow * r, nend = nbeg + len1;
        if (nrow < count) row_issue<G, I16>(Wd4, idx4, nbeg, nend, (nbeg >> 2) + sub, nxt);
        const uint32_t len2 = nrow + stride < count ? nnz[nrow + stride] : 0u;
        float a[W][4] = {};
        if (row < count && end > beg) {
            const uint64_t qlast = (end - 1) >> 2;
            uint64_t q0 = (beg >> 2) + sub;
            row_consume<G, I16, W == 1>(cur, beg, end, q0, xs, a, xpitch);
            for (q0 += 4 * G; q0 <= qlast; q0 += 4 * G) {        // rows longer than one pass
                RowLoads<I16> more;
                row_issue<G, I16>(Wd4, idx4, beg, end, q0, more);
                row_consume<G, I16, W == 1>(more, beg, end, q0, xs, a, xpitch);
            }
        }
        const float b = sub == 0 && row < count && bias ? bias[row] : 0.0f;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const float s = group_sum<G>((a[j][0] + a[j][1]) + (a[j][2] + a[j][3]));
            if (sub == 0 && row < count) {
                float v = b + s;
                if (MM) v = act == SO_ACT_RELU ? so_epilogue<SO_ACT_RELU>(v) : act == SO_ACT_SIGMOID ? so_epilogue<SO_ACT_SIGMOID>(v)
                          : act == SO_ACT_TANH ? so_epilogue<SO_ACT_TANH>(v) : v;
                if constexpr (TELL) {
                    lds_x[(XLDS ? n : 0u) + held] = v;      // behind x: the workgroup's 16 RPW consecutive rows of each pass
                } else y[!MM ? row : W > 1 ? (size_t)row * W + j : (size_t)row * C + blockIdx.y] = v;
            }
        }
        cur = nxt;
        beg = nbeg;
        end = nend;
        len1 = len2;
        held += kWavesPerBlock * RPW;
    }
    tell_host<TELL>(tell, lds_x + (XLDS ? n : 0u), kWavesPerBlock * RPW, stride, blockIdx.x * (kWavesPerBlock * RPW), count, 0u);
}

// Rows of at most G*T nonzeros, G lanes per row.  Such a row is a chain of memory round trips and
// nothing else, so all of a group's first row is requested before x is staged.
template <bool XLDS, bool TELL, int G, int T, typename IdxT>
__device__ __forceinline__ void short_rows(const float *__restrict__ Wd, const IdxT *__restrict__ idx,
                                           const uint2 *__restrict__ rows, uint32_t count, uint32_t block, uint32_t blocks,
                                           uint32_t r, const float *__restrict__ x, uint32_t n, float *lds_x,
                                           const float *__restrict__ bias, float *__restrict__ y, const Tell &tell, float *held, uint32_t at)
{
    const uint32_t sub = threadIdx.x % G;
    const uint32_t stride = blocks * (kBlock / G);
    uint32_t g = block * (kBlock / G) + threadIdx.x / G;
    const uint2 e = g < count ? rows[g] : make_uint2(0u, 0u);
    uint2 en = g + stride < count ? rows[g + stride] : make_uint2(0u, 0u);     // the group's next task, a row ahead
    const uint64_t base = (uint64_t)e.x * r;
    float w[T];
    uint32_t c[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t j = sub + G * t;
        w[t] = j < e.y ? Wd[base + j] : 0.0f;
        c[t] = j < e.y ? idx[base + j] : 0u;
    }
    const float *xs = stage_x<XLDS>(x, n, lds_x);
    if (g < count) {
        float a = 0.0f;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const float xv = sub + G * t < e.y ? xs[c[t]] : 0.0f;      // x may be null when nothing is stored
            a = __builtin_fmaf(w[t], xv, a);
        }
        for (uint32_t j = sub + G * T; j < e.y; j += G) a = __builtin_fmaf(Wd[base + j], xs[idx[base + j]], a);
        a = group_sum<G>(a);
        if (sub == 0) (TELL ? held[threadIdx.x / G] : y[e.x]) = (bias ? bias[e.x] : 0.0f) + a;
    }
    uint32_t place = threadIdx.x / G;
    for (g += stride; g < count; g += stride) {
        const uint2 ec = en;
        if (g + stride < count) en = rows[g + stride];
        const float s = group_row_dot<G>(Wd, idx, (uint64_t)ec.x * r, ec.y, xs, sub);
        place += kBlock / G;
        if (sub == 0) (TELL ? held[place] : y[ec.x]) = (bias ? bias[ec.x] : 0.0f) + s;
    }
    tell_host<TELL>(tell, held, kBlock / G, stride, block * (kBlock / G), count, at);
}

struct BinArgs {
    const uint2 *rowswg, *rows64, *rows16, *rows4;   // (row, nonzeros of the row) per length class
    uint32_t nwg, n64, n16, n4;                      // rows per class
    uint32_t bwg, b64, b16;                          // workgroups given to the workgroup-, 64- and 16-lane classes
};

constexpr uint32_t kBinnedTailBytes = 64;            // behind x in LDS: the 16 waves' partial sums of a workgroup-wide row

template <bool XLDS, bool I16, bool TELL>
__global__ __launch_bounds__(kBlock, TELL ? 4 : 8)          // 64 registers: two workgroups per compute unit (TELL would spill)
void matvec_binned_kernel(const float *__restrict__ Wd, const void *__restrict__ idxv, BinArgs ba, uint32_t r,
                          const float *__restrict__ x, uint32_t n,
                          const float *__restrict__ bias, float *__restrict__ y, Tell tell)
{
    extern __shared__ float lds_x[];
    // TELL: the result in the classes' order, the longest first
    float *const held = lds_x + (XLDS ? ((n + 3u) & ~3u) : 0u) + kBinnedTailBytes / sizeof(float);
    uint32_t b = blockIdx.x;
    if (b < ba.bwg) {
        // Rows of more than 4096 nonzeros: the 16 waves take the row's passes of 1024 slots in turn,
        // the 16 partial sums meet in LDS (behind x) and are added in wave order.
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const f32x4 *Wd4 = reinterpret_cast<const f32x4 *>(Wd);
        const typename ColGroup<I16>::T *idx4 = reinterpret_cast<const typename ColGroup<I16>::T *>(idxv);
        float *part = lds_x + (XLDS ? ((n + 3u) & ~3u) : 0u);
        const float *xs = stage_x<XLDS>(x, n, lds_x);
        for (uint32_t g = b; g < ba.nwg; g += ba.bwg) {
            const uint2 e = ba.rowswg[g];
            const uint64_t beg = (uint64_t)e.x * r, end = beg + e.y;
            const uint64_t qlast = (end - 1) >> 2;                  // e.y > 4096
            float a[1][4] = {};
            for (uint64_t q = (beg >> 2) + wave * 256u + lane; q <= qlast; q += 256u * kWavesPerBlock) {
                RowLoads<I16> L;
                row_issue<64, I16>(Wd4, idx4, beg, end, q, L);
                row_consume<64, I16, false>(L, beg, end, q, xs, a);
            }
            const float s = group_sum<64>((a[0][0] + a[0][1]) + (a[0][2] + a[0][3]));
            if (lane == 0) part[wave] = s;
            __syncthreads();
            if (threadIdx.x == 0) {
                float t = part[0];
#pragma unroll
                for (int w = 1; w < kWavesPerBlock; ++w) t += part[w];
                (TELL ? held[g / ba.bwg] : y[e.x]) = (bias ? bias[e.x] : 0.0f) + t;
            }
            __syncthreads();                                        // part[] is reused by the next row
        }
        tell_host<TELL>(tell, held, 1u, ba.bwg, b, ba.nwg, 0u);
        return;
    }
    b -= ba.bwg;
    if (b < ba.b64) {
        // A wave's first row (its only one unless the class has more rows than the launch has waves):
        // where it is and how long comes in one load, issued before x is staged.  The row itself is
        // requested after the staging: asked for earlier, it delays x (loads return to a wave in
        // order) and with it the barrier; measured 1.3 us slower on the Zipf matrix.
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t stride = ba.b64 * kWavesPerBlock;
        const f32x4 *Wd4 = reinterpret_cast<const f32x4 *>(Wd);
        const typename ColGroup<I16>::T *idx4 = reinterpret_cast<const typename ColGroup<I16>::T *>(idxv);
        uint32_t g = __builtin_amdgcn_readfirstlane(b * kWavesPerBlock + (threadIdx.x >> 6));
        const uint2 e = g < ba.n64 ? ba.rows64[g] : make_uint2(0u, 0u);
        // the wave's next task, requested a row ahead so that its row never waits for it
        uint2 en = g + stride < ba.n64 ? ba.rows64[g + stride] : make_uint2(0u, 0u);
        const uint64_t beg = (uint64_t)e.x * r, end = beg + e.y;
        const uint64_t q0 = (beg >> 2) + lane;
        const float *xs = stage_x<XLDS>(x, n, lds_x);
        RowLoads<I16> A;
        if (e.y > 0) row_issue<64, I16>(Wd4, idx4, beg, end, q0, A);
        if (g < ba.n64) {
            float a[1][4] = {};
            if (e.y > 0) {
                row_consume<64, I16, false>(A, beg, end, q0, xs, a);
                const uint64_t qlast = (end - 1) >> 2;
                for (uint64_t q = q0 + 256; q <= qlast; q += 256) {
                    RowLoads<I16> L;
                    row_issue<64, I16>(Wd4, idx4, beg, end, q, L);
                    row_consume<64, I16, false>(L, beg, end, q, xs, a);
                }
            }
            const float s = group_sum<64>((a[0][0] + a[0][1]) + (a[0][2] + a[0][3]));
            if (lane == 0) (TELL ? held[threadIdx.x >> 6] : y[e.x]) = (bias ? bias[e.x] : 0.0f) + s;
        }
        uint32_t place = threadIdx.x >> 6;
        for (g += stride; g < ba.n64; g += stride) {
            const uint2 ec = en;
            if (g + stride < ba.n64) en = ba.rows64[g + stride];
            const uint64_t nbeg = (uint64_t)ec.x * r;
            const float s = wave_row_dot<I16>(Wd4, idx4, nbeg, nbeg + ec.y, xs, lane);
            place += kWavesPerBlock;
            if (lane == 0) (TELL ? held[place] : y[ec.x]) = (bias ? bias[ec.x] : 0.0f) + s;
        }
        tell_host<TELL>(tell, held, kWavesPerBlock, stride, b * kWavesPerBlock, ba.n64, ba.nwg);
    } else if (b < ba.b64 + ba.b16) {
        const typename ColGroup<I16>::E *idx = reinterpret_cast<const typename ColGroup<I16>::E *>(idxv);
        short_rows<XLDS, TELL, 16, 8>(Wd, idx, ba.rows16, ba.n16, b - ba.b64, ba.b16, r, x, n, lds_x, bias, y, tell, held, ba.nwg + ba.n64);
    } else {
        const typename ColGroup<I16>::E *idx = reinterpret_cast<const typename ColGroup<I16>::E *>(idxv);
        short_rows<XLDS, TELL, 4, 4>(Wd, idx, ba.rows4, ba.n4, b - ba.b64 - ba.b16, gridDim.x - ba.bwg - ba.b64 - ba.b16, r, x, n,
                               lds_x, bias, y, tell, held, ba.nwg + ba.n64 + ba.n16);
    }
}

template <bool XLDS, typename IdxT>
__global__ __launch_bounds__(kBlock)
void matvec_slot_kernel(const float *__restrict__ WdT, const IdxT *__restrict__ idxT,
                        const uint32_t *__restrict__ nnz, uint32_t m,
                        const float *__restrict__ x, uint32_t n,
                        const float *__restrict__ bias, float *__restrict__ y)
{
    extern __shared__ float lds_x[];
    const float *xs = stage_x<XLDS>(x, n, lds_x);
    const uint32_t stride = gridDim.x * kBlock;
    for (uint32_t row = blockIdx.x * kBlock + threadIdx.x; row < m; row += stride) {
        const uint32_t cnt = nnz[row];
        float a = bias ? bias[row] : 0.0f;
        for (uint32_t k = 0; k < cnt; ++k) {
            const size_t e = (size_t)k * m + row;
            a = __builtin_fmaf(WdT[e], xs[idxT[e]], a);
        }
        y[row] = a;
    }
}

// LDS staging of x is worth its per-workgroup copy only when a workgroup then
// serves many nonzeros from it; it needs n floats of LDS (set up once per kernel).
template <typename K>
bool use_lds(so_ctx *ctx, K kernel, uint32_t n, uint64_t nnz_total, uint32_t blocks, size_t extra = 0)
{
    const size_t lds = (size_t)n * sizeof(float) + extra;
    if (n == 0 || lds > (size_t)ctx->max_lds_bytes) return false;
    if (nnz_total < (uint64_t)n * blocks) return false;   // fewer gathers than staged elements
    if (lds > 48 * 1024 && so_allow_big_lds(ctx, (const void *)kernel) != hipSuccess) return false;
    return true;
}

// The row kernel on the row-major arrays, on the 16-bit columns when the handle has them: the C columns of X in turn (MM), or W = C at once, where that
// is the better way; false: it is not.  TELL: also where the results held for the host take the place that x would have in LDS, as launch_bins does (40 874 columns,
// 5236 rows at 94 % sparse from host arrays 81.8 us with x outside LDS, 42.8 with a kernel for the way back).
//
// At once a workgroup streams its rows once and stages all columns, in turn each column has workgroups of its own: better while those fit the chip, whose
// compute units would stand idle otherwise.  Us, in turn / at once, two and three columns: 200 x 3000 at 80 % sparse 4.2 / 4.8 and 4.3 / 5.3, 1000 x 1000 at 70 %
// 4.0 / 4.3 and 4.1 / 4.8, 2000 x 4000 at 90 % 5.0 / 4.9 and 8.6 / 5.4, 4096 x 4096 at 90 % 8.8 / 5.3 and 12.3 / 5.9, 2500 x 12 000 at 90 % 16.4 / 8.9 and 18.4 / 10.1.
template <int W, bool MM, bool TELL>
bool launch_rows(so_ctx *ctx, const so_ellpack *E, const float *dx, uint32_t C, const float *dBias, float *dy, int act, const Tell &tell)
{
    const uint32_t cus = (uint32_t)ctx->compute_units;
    const size_t held = TELL ? kBlock * sizeof(float) : 0, more_x = (size_t)(W - 1) * E->n * sizeof(float), lds = (size_t)E->n * sizeof(float) + more_x + held;
    const bool i16 = E->d_idx16 != nullptr && ctx->tune.matvec_idx16 != 0;
    const void *cols = i16 ? (const void *)E->d_idx16 : (const void *)E->d_idx;
    // Lanes per row by the longest row (one pass of 16 G slots should cover it), but never so
    // few that compute units are left without rows.
    uint32_t G = E->max_nnz <= 128 ? 8u : E->max_nnz <= 256 ? 16u : E->max_nnz <= 512 ? 32u : 64u;
    if (ctx->tune.matvec_lanes) G = (uint32_t)ctx->tune.matvec_lanes;
    else
        while (G < 64 && so_ceil_div(E->m, kWavesPerBlock * (64u / G)) < cus) G *= 2;
    // One resident workgroup per compute unit (the pipelined rows need the registers); each of
    // its 16 waves keeps two passes' loads in flight.
    const uint32_t blocks = std::max(1u, std::min(so_ceil_div(E->m, kWavesPerBlock * (64u / G)), cus));
    if (W > 1 && blocks * C <= cus) return false;
    // The first rows up to their pitch: 0.03 to 0.13 us of 3.7 (40 x 600, 200 x 3000), but up to a quarter more bytes where a wave has one row (8559 x 9895 at 97 %
    // sparse 13.35 -> 13.66 us): up to half a million slots.
    const uint32_t whole = (uint64_t)E->m * E->r <= (1u << 19) ? 1u : 0u;
#define SO_MV_ROWS(G, I16)                                                                                         \
    do {                                                                                                       \
        if (use_lds(ctx, matvec_rows_kernel<true, G, I16, W, MM, TELL>, E->n, E->total_nnz, blocks, more_x + held)) \
            matvec_rows_kernel<true, G, I16, W, MM, TELL><<<dim3(blocks, C / W), kBlock, lds, ctx->stream>>>(E->d_Wd, cols, E->d_nnz, E->m, E->r, \
                                                                                   dx, E->n, dBias, dy, C, act, whole, tell); \
        else if constexpr (W > 1) return false;                                                                \
        else {                                                                                                 \
            if (TELL && use_lds(ctx, matvec_rows_kernel<true, G, I16, W, MM, TELL>, E->n, E->total_nnz, blocks)) return false; \
            matvec_rows_kernel<false, G, I16, W, MM, TELL><<<dim3(blocks, C), kBlock, held, ctx->stream>>>(E->d_Wd, cols, E->d_nnz, E->m, E->r,  \
                                                                                  dx, E->n, dBias, dy, C, act, whole, tell);  \
        }                                                                                                      \
    } while (0)
#define SO_MV_ROWS_G(I16)                                                                                          \
    do {                                                                                                       \
        if (G == 8) SO_MV_ROWS(8, I16);                                                                        \
        else if (G == 16) SO_MV_ROWS(16, I16);                                                                 \
        else if (G == 32) SO_MV_ROWS(32, I16);                                                                 \
        else SO_MV_ROWS(64, I16);                                                                              \
    } while (0)
    if (i16) SO_MV_ROWS_G(true);
    else SO_MV_ROWS_G(false);
#undef SO_MV_ROWS_G
#undef SO_MV_ROWS
    return true;
}

// The length classes in one launch; false: nothing to launch, or TELL has no room for both x and the results in LDS.
template <bool TELL>
bool launch_bins(so_ctx *ctx, const so_ellpack *E, const float *dx, const float *dBias, float *dy, const Tell &tell)
{
    const uint32_t cus = (uint32_t)ctx->compute_units;
    const size_t held = TELL ? kBlock * sizeof(float) : 0, lds = (size_t)E->n * sizeof(float);
    const bool i16 = E->d_idx16 != nullptr && ctx->tune.matvec_idx16 != 0;
    const void *cols = i16 ? (const void *)E->d_idx16 : (const void *)E->d_idx;
    // One launch over the four length classes.  bins[] is ordered 4, 16, 64 lanes, workgroup.
    BinArgs ba;
    ba.rowswg = reinterpret_cast<const uint2 *>(E->bins[3].d_rows);  ba.nwg = E->bins[3].count;
    ba.bwg = std::min(ba.nwg, cus);
    ba.rows4 = reinterpret_cast<const uint2 *>(E->bins[0].d_rows);   ba.n4 = E->bins[0].count;
    ba.rows16 = reinterpret_cast<const uint2 *>(E->bins[1].d_rows);  ba.n16 = E->bins[1].count;
    ba.rows64 = reinterpret_cast<const uint2 *>(E->bins[2].d_rows);  ba.n64 = E->bins[2].count;
    ba.b64 = std::min(so_ceil_div(ba.n64, kWavesPerBlock), 2u * cus);
    ba.b16 = std::min(so_ceil_div(ba.n16, kBlock / 16), std::max(1u, cus / 4));
    const uint32_t b4 = std::min(so_ceil_div(ba.n4, kBlock / 4), std::max(1u, cus / 4));
    // Staging x pays while a workgroup gathers at least as many elements as it stages (use_lds): rather than
    // give that up, a launch with few nonzeros per workgroup takes fewer workgroups of the wave-per-row class,
    // down to one per compute unit (8192 rows of 820 nonzeros: 20.8 us unstaged on 512 workgroups).
    if (E->n > 0) {
        const uint64_t pays = E->total_nnz / E->n;                       // workgroups for which staging pays
        const uint32_t others = ba.bwg + ba.b16 + b4;
        if ((uint64_t)others + ba.b64 > pays && ba.b64 > cus)
            ba.b64 = (uint32_t)std::max<uint64_t>(cus, pays > others ? pays - others : 0);
    }
    const uint32_t blocks = ba.bwg + ba.b64 + ba.b16 + b4;
    if (blocks == 0) return false;
    // TELL: a workgroup holds the results of all its passes, a thread each
    if (TELL && (ba.nwg > ba.bwg * kBlock || ba.n64 > ba.b64 * kBlock || ba.n16 > ba.b16 * kBlock || ba.n4 > b4 * kBlock)) return false;
    // x padded to whole 16-byte groups, then the partial sums of a workgroup-wide row
    const size_t lds_tail = (((size_t)E->n + 3) & ~(size_t)3) * sizeof(float) + kBinnedTailBytes + held;
#define SO_MV_BINNED(I16) \
    do { \
        if (use_lds(ctx, matvec_binned_kernel<true, I16, TELL>, E->n, E->total_nnz, blocks, lds_tail - lds)) \
            matvec_binned_kernel<true, I16, TELL><<<blocks, kBlock, lds_tail, ctx->stream>>>(E->d_Wd, cols, ba, E->r, \
                                                                                       dx, E->n, dBias, dy, tell); \
        else { \
            if (TELL && use_lds(ctx, matvec_binned_kernel<true, I16, TELL>, E->n, E->total_nnz, blocks, lds_tail - lds - held)) return false; \
            matvec_binned_kernel<false, I16, TELL><<<blocks, kBlock, kBinnedTailBytes + held, ctx->stream>>>( \
                E->d_Wd, cols, ba, E->r, dx, E->n, dBias, dy, tell); \
        } \
    } while (0)
    if (i16) SO_MV_BINNED(true);
    else SO_MV_BINNED(false);
#undef SO_MV_BINNED
    return true;
}

} // namespace

so_status so_matvec_columns(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    if (C == 2u && launch_rows<2, true, false>(ctx, E, dX, C, dBias, dY, act, Tell())) return SO_OK;
    if (C == 3u && launch_rows<3, true, false>(ctx, E, dX, C, dBias, dY, act, Tell())) return SO_OK;
    launch_rows<1, true, false>(ctx, E, dX, C, dBias, dY, act, Tell());
    return SO_OK;
}

// The layout of a launch that leaves it to the library.
static int choose_layout(const so_ctx *ctx, const so_ellpack *E)
{
    // Length classes for skewed rows (the widest row far above the mean).  For even rows the row kernel, which
    // requests a wave's next row while it sums the current one, is the better one except on 16-bit columns
    // where the length-class launch fills its two workgroups per compute unit with two or three rows per wave
    // (16384 columns, 820 nonzeros per row; rows / us row kernel / us length classes: 8192 / 9.3 / 10.1,
    // 16384 / 15.6 / 15.0, 24576 / 21.7 / 21.7, 32768 / 27.5 / 28.3, 49152 / 39.3 / 42.4, 65536 / 51 / 56).
    const bool skewed = (uint64_t)E->r * E->m > 2 * E->total_nnz + E->m;
    const uint32_t per_wave_x2 = E->m / (16u * (uint32_t)ctx->compute_units);           // rows per wave of 2 x CUs workgroups, doubled
    const bool few_rows = E->d_idx16 != nullptr && ctx->tune.matvec_idx16 != 0 && per_wave_x2 >= 4 && per_wave_x2 < 6;
    if ((E->layouts & SO_LAYOUT_BINS) && (skewed || few_rows)) return SO_LAYOUT_BINS;
    if ((E->layouts & SO_LAYOUT_SLOT) && E->max_nnz <= 64) return SO_LAYOUT_SLOT;
    return SO_LAYOUT_ROW;
}

extern "C" so_status so_matvec(so_ctx *ctx, const so_ellpack *E, const float *dx,
                               const float *dBias, float *dy, int layout)
{
    SO_REQUIRE(ctx && E, "so_matvec: null argument");
    if (E->m == 0) return SO_OK;
    SO_REQUIRE(dy != nullptr, "so_matvec: y is null");
    SO_REQUIRE(dx != nullptr || E->total_nnz == 0, "so_matvec: x is null");
    if (layout == 0) layout = choose_layout(ctx, E);
    SO_REQUIRE(layout == SO_LAYOUT_ROW || layout == SO_LAYOUT_SLOT || layout == SO_LAYOUT_BINS,
               "so_matvec: unknown layout %d", layout);
    SO_REQUIRE((E->layouts & layout) != 0, "so_matvec: layout %d was not uploaded", layout);

    const uint32_t cus = (uint32_t)ctx->compute_units;
    const size_t lds = (size_t)E->n * sizeof(float);
    if (layout == SO_LAYOUT_ROW) {
        launch_rows<1, false, false>(ctx, E, dx, 1, dBias, dy, SO_ACT_NONE, Tell());
    } else if (layout == SO_LAYOUT_SLOT) {
        const uint32_t blocks = std::max(1u, std::min(so_ceil_div(E->m, kBlock), 2u * cus));
#define SO_MV_SLOT(T, COLS)                                                                                        \
        do {                                                                                                       \
            if (use_lds(ctx, matvec_slot_kernel<true, T>, E->n, E->total_nnz, blocks))                             \
                matvec_slot_kernel<true, T><<<blocks, kBlock, lds, ctx->stream>>>(E->d_WdT, COLS, E->d_nnz, E->m,  \
                                                                                  dx, E->n, dBias, dy);            \
            else                                                                                                   \
                matvec_slot_kernel<false, T><<<blocks, kBlock, 0, ctx->stream>>>(E->d_WdT, COLS, E->d_nnz, E->m,   \
                                                                                 dx, E->n, dBias, dy);             \
        } while (0)
        if (E->d_idxT16 && ctx->tune.matvec_idx16 != 0) SO_MV_SLOT(uint16_t, E->d_idxT16);
        else SO_MV_SLOT(uint32_t, E->d_idxT);
#undef SO_MV_SLOT
    } else if (!launch_bins<false>(ctx, E, dx, dBias, dy, Tell())) return SO_OK;
    SO_LAUNCH_CHECK();
    return SO_OK;
}

// The result straight into the staging memory, one launch fewer in a chain that is nothing but launches and the link.  ellpack_matvec from
// host arrays, us, a kernel for the way back / this: 1500 x 1000 at 90 % sparse 17.9 / 15.1, 2864 x 3084 at 97 % 19.3 / 16.1, 4096 x 4096 at 80 %
// 21.6 / 17.6, 8000 x 2000 at 90 % 23.6 / 21.2; Zipf rows 1077 x 3800 19.4 / 15.8, 4096 x 4096 20.2 / 17.4.  Beyond kStagePairsMost rows the host's look at each
// pair, and in the classes' order its walk over y, take longer than the launch did: 16384 x 2000 29.0 / 32.7, 12000 x 2000 with Zipf rows 24.2 / 26.3.
extern "C" so_status so_matvec_to_host(so_ctx *ctx, const so_ellpack *E, const float *dx, const float *dBias, float *dy, float *y, int layout)
{
    SO_REQUIRE(ctx && E, "so_matvec_to_host: null argument");
    if (E->m == 0) return SO_OK;
    SO_REQUIRE(y != nullptr && dy != nullptr, "so_matvec_to_host: y is null");
    SO_REQUIRE(!ctx->capturing, "so_matvec_to_host: not allowed while a graph is being recorded");
    const int kernel = layout == 0 ? choose_layout(ctx, E) : layout;
    const bool rows = kernel == SO_LAYOUT_ROW, bins = kernel == SO_LAYOUT_BINS && (E->layouts & SO_LAYOUT_BINS) && E->bin_order.size() == E->m;
    Tell tell;
    if ((rows || bins) && (dx != nullptr || E->total_nnz == 0) && so_stage_result(ctx, E->m, &tell.rows, &tell.turn)) {
        bool told = false;
        if (rows ? launch_rows<1, false, true>(ctx, E, dx, 1, dBias, nullptr, SO_ACT_NONE, tell) : launch_bins<true>(ctx, E, dx, dBias, nullptr, tell)) {
            SO_LAUNCH_CHECK();
            const so_status s = so_stage_result_take(ctx, E->m, rows ? nullptr : E->bin_order.data(), y, tell.turn, &told);
            if (s != SO_OK || told) return s;
        }
    }
    const so_status s = so_matvec(ctx, E, dx, dBias, dy, layout);
    return s != SO_OK ? s : so_stage_out(ctx, y, dy, (size_t)E->m * sizeof(float));
}
