// Bf16-planes matmul: Y = act(E X + bias) as a dense product on the bf16 matrix cores in fp32 precision, part of layout
// SO_LAYOUT_RBM.
//
// A float is the exact sum of three bf16 numbers, hi + mid + lo (8 significant bits each, rounded to nearest, the next one
// holding what the last left).  The matrix is kept as three bf16 planes, zeros included, in the order in which
// v_mfma_f32_32x32x16_bf16 reads its operand; X is split on its way into LDS.  Of the nine products of planes the six
// whose size may be 2^-17 of the whole or more are added up.  What the other three leave out is at most 2^-24 of the product (where both
// factors are near 1 + 2^-8 - 2^-17 times a power of two), as much as one fp32 rounding, and 2^-27.5 in the 2-norm over all mantissas.
// hi * hi goes to one set of accumulators and the five small products (2^-7 of it at most) to another, so that the large sums are
// rounded once per 16 columns, and every 512 columns they are added to totals in LDS.  So long sums are closer than a chain of fmaf, but an output of a
// single nonzero may be 1.7 x 2^-24 off instead of 2^-24.
//
// Why: an MFMA of 32 x 32 x 16 takes a SIMD 32 clocks, so six of them do 85 fp32 multiply-adds per clock on zeros and
// nonzeros alike.  The quad-union kernel (matmul_quad.hip) does 32 per clock on the union of four rows, which is 59 % of
// the matrix at 80 % sparsity, 76 % at 70 %, 94 % at 50 %; the row-block-merged kernel (matmul_rbm.hip) pays per nonzero.
//
// What bounds it: the matrix cores.  An iteration -- 128 rows x 64 columns x 64 of K, 48 MFMAs on each SIMD, 1536 clocks --
// takes 0.87 us while half of the compute units are at work (2090 clocks at 2.4 GHz: the rest is the barrier, first LDS reads
// and the instructions of the splitting, seven per value of X) and 1.2 on the whole chip, whose clock falls to 1.7 GHz
// under bf16 MFMAs.  Beside that 4 us of launch, first loads and first split, and 2.4 to 4.8 for the exchange of partial
// tiles between two to five workgroups.  With eight waves that all split and multiply in turn an iteration took 1.4 to 1.5
// us, with four waves splitting 0.93.  128 x 64 per workgroup against 64 x 128 has half the values of X to split: 18.4
// against 19.4 us (3001 x 2777 x 101) and 42.7 against 47.2 (4096 x 4096 x 256).
//
// Measured, one handle launched again and again, before and now: 3001 x 2777 x 101 at 70 % sparse 27.1 (row-block-merged)
// and 18.5 to 20 us on different cards; 4096 x 4096 x 256 at 70 % 60.7 (row-block-merged) and 43.9, at 50 % 84.1 (quad-union)
// and 45.2 (191 TFLOP/s counting the zeros).  Error in the 2-norm against 64 bits: 8.9e-8 (1.1e-7 before), 9.2e-8
// (1.5e-7), 1.1e-7 (4.1e-7).
#include "so_internal.h"
#include "lds_sync.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>

namespace {

constexpr uint32_t MULTIPLIERS = 256, SPLITTERS = 512, THREADS = MULTIPLIERS + SPLITTERS;
constexpr uint32_t FRAG = 1024;                         // bytes of one operand of an MFMA: 64 lanes x 8 bf16
constexpr uint32_t STEPS = 4, KI = 16 * STEPS;          // an iteration: runs of 16 columns of the matrix
constexpr uint32_t BM = 128, BN = 64, NT = BN / 32;     // a workgroup's rows and dense columns
constexpr uint32_t BUF = STEPS * NT * 3 * FRAG;         // LDS of one iteration's X
constexpr uint32_t SPILL = 8;                           // iterations after which the large sums leave their registers
constexpr uint32_t SUMS_AT = 2 * BUF, KEPT_AT = SUMS_AT + BM * BN * 4, FLAGS_AT = KEPT_AT + BM * BN * 4, LDS_BYTES = FLAGS_AT + 16;
static_assert(SPLITTERS == KI / 8 * BN, "a splitting thread takes one column's group of 8 rows");
constexpr uint32_t kMostColumns = (1u << 24) - 1u;      // a row tile's planes, 192 bytes per column, are addressed with 32 bits
static_assert(((uint64_t)kMostColumns + KI) / 16 * 3 * FRAG <= 0xffffffffull, "offsets into a row tile's planes");

// The planes hold X times 2^24 and the matrix times 2^-24: then the last bit of any float of X, 2^-149, is a bf16 of normal size, and so
// is that of any weight from kLeastWeight on.  A pass for large values takes X times 2^-64.  With weights of at most kMostWeight and fewer than
// 2^24 columns no sum of values below kLarge, nor of large ones scaled down, leaves the range: 24 + 39 + 40 bits, 24 + 39 - 24 + 128 - 64.
constexpr float kUp = 0x1p24f, kLarge = 0x1p40f, kLargeDown = 0x1p-88f, kMostWeight = 0x1p39f, kLeastWeight = 0x1p-76f;

// The passes of a workgroup over its range of K: ordinarily the first alone.
enum Pass : uint32_t { ALL, SMALL, LARGE, NOT_FINITE };
// flags[ALL] asks for the others, flags[LARGE] and flags[NOT_FINITE] say whether there is anything to do in them.
__device__ __forceinline__ uint32_t next_pass(uint32_t pass, const uint32_t *flags)
{
    const auto set = [&](uint32_t p) { return __builtin_amdgcn_readfirstlane(flags[p]) != 0u; };
    if (pass == ALL) return set(ALL) ? SMALL : ALL;
    if (pass == SMALL && set(LARGE)) return LARGE;
    return pass != NOT_FINITE && set(NOT_FINITE) ? NOT_FINITE : ALL;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct PlanesArgs {
    const char *A;              // [row tile of 32][16 columns][plane][FRAG]
    uint32_t m, n, C, k16;      // k16: runs of 16 columns kept per row tile
    uint32_t ks, iters, iters_per, nslab, mbs, per_xcd;
    const float *X, *bias;
    float *Y, *part;
    uint32_t *counters;
};

// Two floats to bf16 (nearest even), the first in the low half; `v` keeps what is left of them.
__device__ __forceinline__ uint32_t take_plane(float &v0, float &v1)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v0, v1}, bf16x2));
    v0 -= __uint_as_float(u << 16);
    v1 -= __uint_as_float(u & 0xffff0000u);
    return u;
}
__device__ __forceinline__ uint32_t last_plane(float v0, float v1)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v0, v1}, bf16x2));
}

// Of two bf16 numbers their signs, as +-1 or 0.
__device__ __forceinline__ uint32_t signs_of(uint32_t pair)
{
    const uint32_t some = (((pair & 0x7fff7fffu) + 0x7fff7fffu) & 0x80008000u) >> 15;      // a bit per number that is not 0
    return some * 0x3f80u | (pair & (some << 15));
}

// A workgroup owns 128 rows x 64 columns and a range of K.  Twelve waves: four multiply, 32 rows x 64 columns each; eight
// fetch X, split it and store the planes in LDS, an iteration of 64 rows of X ahead (two buffers, a barrier per iteration).
// A SIMD has one of the former and two of the latter, so that the splitting's vector instructions run in the shadow of
// the MFMAs.
//
// Values that the scaled planes cannot hold -- infinities, NaNs and finite ones from 2^104 on -- come out of the splitting as NaN, and sums
// that overflow do not come out finite.  The workgroup then goes over its range of K again: with the values below 2^40
// alone, with the finite ones above it alone (scaled down), and for infinities and NaNs with the signs of the matrix, counting in whole
// numbers what an output receives: as many of one sign as in all is an infinity, otherwise a NaN.  A zero of the matrix meets none of them.
// Us with ordinary values, with an infinity in one column, an infinity or a NaN in each, 1e32 in each: 3001 x 2777 x 101 at 70 % 21, 43, 44, 46 (the
// row-block-merged kernel 29 with any); 4096 x 4096 x 256 at 50 % 49, 106, 122, 129 (the quad-union kernel 97, 197, 2380, 92).  Tiny
// values cost nothing.  (Giving up every column with one of these, or with a nonzero value below 2^-110, and summing its outputs
// over the nonzeros took 98 with one such column, 4660 with one such value in each; 240 and 14 400.)
template <int ACT>
__global__ __launch_bounds__(THREADS)
void ellpack_matmul_planes_kernel(PlanesArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t *flags = reinterpret_cast<uint32_t *>(lds + FLAGS_AT);  // by pass; [SMALL]: the arrival word
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup ids go round the 8 XCDs; an XCD takes a contiguous share of the (K part, row block, slab) triples, so that
    // it touches one or two parts of X and the slabs of a row block share its L2.
    const uint32_t id = (blockIdx.x & 7u) * a.per_xcd + (blockIdx.x >> 3), tiles = a.mbs * a.nslab;
    if ((blockIdx.x >> 3) >= a.per_xcd || id >= tiles * a.ks) return;
    const uint32_t kp = id / tiles, tile = id - kp * tiles, mb = tile / a.nslab, slab = tile - mb * a.nslab;
    const uint32_t it0 = kp * a.iters_per, count = min(a.iters, it0 + a.iters_per) - it0;
    if (tid < 4u) flags[tid] = 0u;

    if (wave >= MULTIPLIERS / 64u) {
        // A thread takes 8 rows of one column, a wave the same rows.  Rows past the last one come as zeros: out of the buffer's range.
        const uint32_t xt = tid - MULTIPLIERS, xc = xt % BN, g = xt / BN, pitch = a.C * 4u, step = KI * pitch;
        uint32_t at[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) at[j] = (g * 8u + j) * pitch + min(slab * BN + xc, a.C - 1u) * 4u;
        u32x4 *const to = reinterpret_cast<u32x4 *>(lds + ((g >> 1) * NT + (xc >> 5)) * 3u * FRAG) + (g & 1u) * 32u + (xc & 31u);
        float x[2][8];
        float odd = 0.0f;                                            // becomes NaN with a value that the planes do not hold
        auto request = [&](int set, uint32_t it) {
            const uint64_t from = (uint64_t)it * step, end = (uint64_t)a.n * pitch;
            const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X) + from / 4u, 0, from < end ? (int)(uint32_t)(end - from) : 0, 0x00020000);
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) x[set][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, (int)at[j], 0, 0));
            __builtin_amdgcn_sched_barrier(0);
        };
        auto split = [&](int set) {
            u32x4 p0, p1, p2;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v0 = x[set][2 * e] * kUp, v1 = x[set][2 * e + 1] * kUp;
                p0[e] = take_plane(v0, v1);
                p1[e] = take_plane(v0, v1);
                p2[e] = last_plane(v0, v1);
                odd = __builtin_elementwise_maximum(odd, __builtin_elementwise_maximum(v0, v1));   // (inf - inf)
            }
            u32x4 *p = to + set * (BUF / 16u);
            p[0] = p0; p[64] = p1; p[128] = p2;
            __builtin_amdgcn_sched_barrier(0);
        };
        auto fill = [&](auto &&put) {
            request(0, it0);
            request(1, it0 + 1u);
            put(0);
            __syncthreads();
            // (nothing in the loops is conditional, so that the compiler's waits leave the younger requests in flight; what they
            // fetch past the end is not used)
            for (uint32_t i = 0; i + 1u < count; i += 2u) {
                request(0, it0 + i + 2u);
                put(1);
                __syncthreads();
                request(1, it0 + i + 3u);
                put(0);
                __syncthreads();
            }
            if (count & 1u) __syncthreads();
        };
        fill(split);
        if (__builtin_isnan(odd)) flags[ALL] = 1u;
        __syncthreads();
#pragma unroll 1
        for (uint32_t pass = next_pass(ALL, flags); __builtin_expect(pass != ALL, 0); pass = next_pass(pass, flags)) {
            bool large = false, not_finite = false;
            fill([&](int set) {
                uint32_t sign[8], any[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v = x[set][j], size = __builtin_fabsf(v);
                    const bool below = size < kLarge, finite = size <= 3.40282347e38f;
                    large |= !below && finite;
                    not_finite |= !finite;
                    any[j] = finite ? 0u : 0x3f80u;
                    sign[j] = finite || __builtin_isnan(v) ? 0u : __float_as_uint(v) >> 31 << 15 | 0x3f80u;
                    x[set][j] = pass == SMALL ? (below ? v : 0.0f) : !below && finite ? v * kLargeDown : 0.0f;
                }
                if (pass != NOT_FINITE) { split(set); return; }
                u32x4 *p = to + set * (BUF / 16u);
                p[0] = u32x4{sign[0] | sign[1] << 16, sign[2] | sign[3] << 16, sign[4] | sign[5] << 16, sign[6] | sign[7] << 16};
                p[64] = u32x4{any[0] | any[1] << 16, any[2] | any[3] << 16, any[4] | any[5] << 16, any[6] | any[7] << 16};
                __builtin_amdgcn_sched_barrier(0);
            });
            if (pass == SMALL && large) flags[LARGE] = 1u;
            if (pass == SMALL && not_finite) flags[NOT_FINITE] = 1u;
            __syncthreads();
        }
        if (a.ks > 1u) { __syncthreads(); __syncthreads(); }
        return;
    }

    f32x4 s[8];                                                      // element i = 4 j + e of tile t: s[4 t + j][e]
    {
        f32x16 big[2], small[2];
        f32x4 *const sums = reinterpret_cast<f32x4 *>(lds + SUMS_AT) + tid, *const kept = reinterpret_cast<f32x4 *>(lds + KEPT_AT) + tid;
        const uint32_t rt = min(mb * 4u + wave, (a.m + 31u) / 32u - 1u);   // row tiles past the last repeat it
        const uint32_t bytes = a.k16 * 3u * FRAG, lane16 = lane * 16u;
        const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(a.A) + (size_t)rt * bytes, 0, (int)bytes, 0x00020000);
        u32x4 w[STEPS][3], x[2][3];
        auto request = [&](int s, uint32_t i) {
            const uint32_t at = ((it0 + min(i, count - 1u)) * STEPS + (uint32_t)s) * (3u * FRAG);
#pragma unroll
            for (int k = 0; k < 3; ++k) w[s][k] = __builtin_amdgcn_raw_buffer_load_b128(ar, (int)(lane16 + k * FRAG), (int)at, 0);
        };
        auto read = [&](uint32_t buf, int s, int t) {
            const u32x4 *xb = reinterpret_cast<const u32x4 *>(lds + buf * BUF + (s * NT + t) * 3u * FRAG) + lane;
#pragma unroll
            for (int k = 0; k < 3; ++k) x[t][k] = xb[k * 64];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto mfma = [](const u32x4 &p, const u32x4 &q, f32x16 &acc) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, p), __builtin_bit_cast(bf16x8, q), acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto clear = [&] {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int k = 0; k < 16; ++k) big[t][k] = small[t][k] = 0.0f;
        };
        auto multiply = [&] {
            clear();
#pragma unroll
            for (int j = 0; j < 8; ++j) sums[j * MULTIPLIERS] = f32x4{0.f, 0.f, 0.f, 0.f};
            // A run's six products of one tile while the other tile's operands come from LDS; the matrix's are requested an
            // iteration ahead, into the registers of the run that is done with.
#pragma unroll
            for (int s = 0; s < (int)STEPS; ++s) request(s, 0u);
            __syncthreads();
            for (uint32_t i = 0; i < count; ++i) {
                const uint32_t buf = i & 1u;
                read(buf, 0, 0);
#pragma unroll
                for (int s = 0; s < (int)STEPS; ++s) {
                    const u32x4 *v = w[s];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        if (t == 0) read(buf, s, 1);
                        else if (s + 1 < (int)STEPS) read(buf, s + 1, 0);
                        mfma(v[2], x[t][0], small[t]); mfma(v[0], x[t][0], big[t]); mfma(v[0], x[t][2], small[t]);
                        mfma(v[1], x[t][1], small[t]); mfma(v[1], x[t][0], small[t]); mfma(v[0], x[t][1], small[t]);
                    }
                    request(s, i + 1u);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // long sums are rounded more often: each lane keeps its totals in LDS
                if (i % SPILL == SPILL - 1u) {
                    f32x4 v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = sums[j * MULTIPLIERS];
#pragma unroll
                    for (int k = 0; k < 32; ++k) { v[k / 4][k % 4] += big[k / 16][k % 16]; big[k / 16][k % 16] = 0.0f; }
#pragma unroll
                    for (int j = 0; j < 8; ++j) sums[j * MULTIPLIERS] = v[j];
                }
                __syncthreads();
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                s[j] = sums[j * MULTIPLIERS];
#pragma unroll
                for (int e = 0; e < 4; ++e) s[j][e] += big[j / 4][j % 4 * 4 + e] + small[j / 4][j % 4 * 4 + e];
            }
        };
        multiply();
        float most = 0.0f;                                           // infinite or NaN where a sum is not finite
#pragma unroll
        for (int k = 0; k < 32; k += 2)
            most = __builtin_elementwise_maximum(most, __builtin_elementwise_maximum(__builtin_fabsf(s[k / 4][k % 4]), __builtin_fabsf(s[k / 4][k % 4 + 1])));
        if (!(most <= 3.40282347e38f)) flags[ALL] = 1u;
        __syncthreads();                                             // the flags
        uint32_t pass = next_pass(ALL, flags);
        if (__builtin_expect(pass != ALL, 0)) {
#pragma unroll 1
            do {
                multiply();
#pragma unroll
                for (int j = 0; j < 8; ++j) kept[j * MULTIPLIERS] = pass == SMALL ? s[j] : kept[j * MULTIPLIERS] + s[j] * (1.0f / kLargeDown);
                __syncthreads();
                pass = next_pass(pass, flags);
            } while (pass == LARGE);
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] = kept[j * MULTIPLIERS];
            if (pass == NOT_FINITE) {
                clear();
                __syncthreads();
#pragma unroll 1
                for (uint32_t i = 0; i < count; ++i) {
#pragma unroll
                    for (int s = 0; s < (int)STEPS; ++s) request(s, i);
#pragma unroll
                    for (int s = 0; s < (int)STEPS; ++s) {
                        u32x4 sign, any;
#pragma unroll
                        for (int k = 0; k < 4; ++k) { sign[k] = signs_of(w[s][0][k]); any[k] = sign[k] & 0x7fff7fffu; }
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            read(i & 1u, s, t);
                            mfma(sign, x[t][0], big[t]);
                            mfma(any, x[t][1], small[t]);
                        }
                    }
                    __syncthreads();
                }
                __syncthreads();
#pragma unroll
                for (int k = 0; k < 32; ++k) {
                    const float signs = big[k / 16][k % 16], all = small[k / 16][k % 16];
                    if (all != 0.0f) s[k / 4][k % 4] = __builtin_fabsf(signs) == all ? __builtin_copysignf(INFINITY, signs) : NAN;
                }
            }
        }
    }
    if (a.ks > 1u) {
        // sc1: written through to memory, whichever XCD the tile's other workgroups run on
        constexpr int SC1 = 16;
        const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(a.part + (size_t)tile * a.ks * 8192u, 0, (int)(a.ks * 32768u), 0x00020000);
#pragma unroll
        for (int j = 0; j < 8; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s[j]), pr, (int)((kp * 8u + j) * 4096u + tid * 16u), 0, SC1);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        __syncthreads();
        if (tid == 0) flags[SMALL] = __hip_atomic_fetch_add(&a.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (flags[SMALL] != a.ks - 1u) return;                          // the last workgroup of the tile to arrive finishes it
        if (tid == 0) __hip_atomic_store(&a.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t k = 0; k < a.ks; k += 2u) {                    // in order; a part past the last comes as zeros
            u32x4 v[2][8];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = __builtin_amdgcn_raw_buffer_load_b128(pr, (int)(((k + i) * 8u + j) * 4096u + tid * 16u), 0, SC1);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) s[j] += __builtin_bit_cast(f32x4, v[i][j]);
        }
    }
    // element (j, e) of a tile: row 8 j + 4 (lane / 32) + e, column lane % 32.  Stores to rows past the last fall out of the
    // buffer's range.
    const uint32_t row0 = (mb * 4u + wave) * 32u, half = lane >> 5, pitch = a.C * 4u;
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.Y, 0, (int)(a.m * pitch), 0x00020000);
    f32x4 bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[j][e] = a.bias ? a.bias[min(row0 + 8u * j + 4u * half + e, a.m - 1u)] : 0.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t c = slab * BN + t * 32u + (lane & 31u);
        if (c >= a.C) continue;
        const uint32_t at = (row0 + 4u * half) * pitch + c * 4u;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(so_epilogue<ACT>(s[4 * t + j][e] + bias[j][e])), yr, (int)(at + (8u * j + e) * pitch), 0, 0);
    }
}

// One stored nonzero per thread into the three planes (which are zeros before).
__global__ __launch_bounds__(256)
void planes_scatter_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx, const uint32_t *__restrict__ nnz, uint32_t m, uint32_t r,
                           uint32_t k16, uint16_t *__restrict__ A)
{
    const uint32_t row = blockIdx.x;
    for (uint32_t s = threadIdx.x; s < nnz[row]; s += 256u) {
        const uint32_t k = idx[(size_t)row * r + s];
        float v = Wd[(size_t)row * r + s] * (1.0f / kUp), zero = 0.0f;
        const uint32_t p0 = take_plane(v, zero), p1 = take_plane(v, zero), p2 = last_plane(v, zero);
        uint16_t *to = A + ((size_t)(row >> 5) * k16 + (k >> 4)) * (3 * FRAG / 2) + ((row & 31u) + ((k >> 3) & 1u) * 32u) * 8u + (k & 7u);
        to[0] = (uint16_t)p0; to[FRAG / 2] = (uint16_t)p1; to[FRAG] = (uint16_t)p2;
    }
}

template <int ACT>
so_status launch(so_ctx *ctx, const PlanesArgs &a, uint32_t blocks)
{
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_matmul_planes_kernel<ACT>));
    ellpack_matmul_planes_kernel<ACT><<<blocks, THREADS, LDS_BYTES, ctx->stream>>>(a);
    return SO_OK;
}

size_t part_bytes(const so_planes_plan &p) { return (size_t)p.mbs * p.nslab * p.ks * BM * BN * sizeof(float); }
size_t counter_bytes(const so_planes_plan &p) { return (size_t)p.mbs * p.nslab * sizeof(uint32_t); }

so_status workspace(so_ctx *ctx, const so_ellpack *E, uint32_t C, const so_planes_plan &p)
{
    if (p.ks == 1) return SO_OK;
    SO_REQUIRE((uint64_t)p.mbs * p.nslab * p.ks < (1ull << 28), "so_matmul: %u x %u output is too large for one launch", E->m, C);
    return so_matmul_workspace(ctx, part_bytes(p), counter_bytes(p));
}

} // namespace

// Workgroups per tile by estimated time (us): rounds of one workgroup per compute unit, an iteration slower where the whole
// chip multiplies (its clock falls), and for a split the exchange of partial tiles; fitted to the launches below.  Measured, us at 1, 2, 3, ... workgroups
// per tile: 3001 x 2777 x 101 42.0, 25.5, 20.7, 18.9, 19.9, 27.7; 4096 x 4096 x 256 60, 43.8, 53, 51; 4096 x 784 x 256 15.6, 15.9, 22.0.
so_planes_plan so_matmul_planes_choose(const so_ctx *ctx, uint32_t m, uint32_t n, uint32_t C)
{
    so_planes_plan best{};
    best.us = 1e30;
    const double cus = ctx->compute_units;
    const uint32_t mbs = so_ceil_div(m, BM), nslab = so_ceil_div(C, BN), iters = so_ceil_div(n, KI);
    for (uint32_t ks = 1; ks <= iters && ks <= so_planes::kMaxSplit; ++ks) {
        const uint32_t per = so_ceil_div(iters, ks), parts = so_ceil_div(iters, per);
        const bool asked = (int)ks == ctx->tune.matmul_planes_split;
        if (parts != ks && !asked) continue;
        const double wgs = (double)mbs * nslab * parts;
        const double us = std::ceil(wgs / cus) * (4.0 + per * (0.87 + 0.75 * std::max(0.0, std::min(1.0, wgs / cus) - 0.55))) + (parts > 1 ? 0.8 + 0.8 * parts : 0.0);
        if (us < best.us || asked) best = so_planes_plan{parts, iters, per, nslab, mbs, us};
        if (asked) break;
    }
    best.us = std::max(best.us, 4.0 + 1.2e-6 * m * n);               // the planes come from memory at 5 TB/s
    return best;
}

so_status so_planes_build(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *nnz)
{
    so_planes &P = E->planes;
    if (!E->ascending || E->total_nnz == 0 || E->n > kMostColumns) return SO_OK;       // (a column named twice by a row has one place)
    // values that have room for three planes and overflow nothing, and no stored zeros (which make NaNs of infinities in X)
    std::atomic<bool> room{true};
    so_parallel(E->m, E->total_nnz, [&](uint32_t i0, uint32_t i1) {
        bool ok = true;
        for (uint32_t i = i0; i < i1 && ok; ++i)
            for (uint32_t k = 0; k < nnz[i]; ++k) {
                const float v = std::fabs(Wd[(size_t)i * E->r + k]);
                ok = ok && v <= kMostWeight && v >= kLeastWeight;
            }
        if (!ok) room = false;
    });
    if (!room) return SO_OK;
    const uint32_t tiles = so_ceil_div(E->m, 32), k16 = so_ceil_div(E->n, KI) * STEPS;
    void *p = nullptr;
    const size_t bytes = (size_t)tiles * k16 * 3 * FRAG;
    so_status s = so_malloc(ctx, bytes, &p);
    if (s != SO_OK) return s;
    P.d_a = p;
    P.k16 = k16;
    SO_HIP(hipMemsetAsync(p, 0, bytes, ctx->stream));
    planes_scatter_kernel<<<E->m, 256, 0, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->m, E->r, k16, (uint16_t *)p);
    SO_LAUNCH_CHECK();
    return SO_OK;
}

void so_planes_free(so_ellpack *E)
{
    if (E->planes.d_a) (void)hipFree(E->planes.d_a);
    E->planes = so_planes();
}

bool so_matmul_planes_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return E->planes.d_a != nullptr && C >= 1 && std::max<uint64_t>(E->n, (uint64_t)E->m + 128) * C * 4u <= 0xffffffffull && (size_t)ctx->max_lds_bytes >= LDS_BYTES;
}

so_status so_matmul_planes_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C) { return workspace(ctx, E, C, so_matmul_planes_choose(ctx, E->m, E->n, C)); }

bool so_matmul_planes_ready(const so_ctx *ctx, const so_planes_plan &p)
{
    return p.ks == 1 || (ctx->mm_part && ctx->mm_counters && part_bytes(p) <= ctx->mm_part->bytes && counter_bytes(p) <= ctx->mm_counters->bytes);
}

so_status so_matmul_planes_launch(so_ctx *ctx, const so_ellpack *E, const so_planes_plan &p, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    const so_status s = workspace(ctx, E, C, p);
    if (s != SO_OK) return s;
    const uint32_t per_xcd = so_ceil_div((uint64_t)p.mbs * p.nslab * p.ks, 8);
    const PlanesArgs a{(const char *)E->planes.d_a, E->m, E->n, C, E->planes.k16, p.ks, p.iters, p.iters_per, p.nslab, p.mbs, per_xcd, dX, dBias, dY,
                       ctx->mm_part ? (float *)ctx->mm_part->p : nullptr, ctx->mm_counters ? (uint32_t *)ctx->mm_counters->p : nullptr};
    const uint32_t blocks = 8u * per_xcd;
    switch (act) {
    case SO_ACT_RELU:    return launch<SO_ACT_RELU>(ctx, a, blocks);
    case SO_ACT_SIGMOID: return launch<SO_ACT_SIGMOID>(ctx, a, blocks);
    case SO_ACT_TANH:    return launch<SO_ACT_TANH>(ctx, a, blocks);
    default:             return launch<SO_ACT_NONE>(ctx, a, blocks);
    }
}
