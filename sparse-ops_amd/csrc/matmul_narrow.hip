// Narrow matmul: Y = act(E X + bias) for up to 32 dense columns, or for few rows, on the quad-union copy of the matrix (matmul_quad.hip,
// layout SO_LAYOUT_RBM).
//
// The quad-union kernel gives 64 lanes 64 columns, four union columns (steps) at a time; with 8 columns seven eighths of its LDS
// reads and MFMAs are for nothing.  Here the 16 blocks of v_mfma_f32_4x4x1_16b_f32 are 16 steps, a chunk, as the copy stores them:
// block b multiplies step b's four weights by four lanes' values of step b's own row of X.  A lane reads V = 1, 2 or 4 values of
// its row at once, so a chunk costs one LDS read and V MFMAs for 4 V columns; for 17 to 32 columns a block pair shares the
// columns and a chunk is two reads of V = 4 (CBSZ 1, ABID 0 and 1).  The sums over the blocks are taken at the end.
//
// Decomposition.  A workgroup of 16 waves owns 1 to 16 quads of rows, as few as give no more workgroups than compute units, and
// the whole of K: all of X (up to 160 KB) is copied to LDS once, one barrier, and from there on a wave only waits for its own
// chunks, which are requested four to eight ahead, the first before X.  No partial tiles are exchanged.  (A matrix whose X does
// not fit stays on the quad-union kernel.)
//
// What bounds it: small launches the latencies of launch (2.5 us) and first loads (1.1); large ones the copy's bytes (4096 x 4096
// x 8, 50 % dense: 65 MB, 16 us, 4.1 TB/s) and, from 17 columns on, bank conflicts of the 128-byte rows.  Copying X in
// two rounds of eight loads cost 1 to 2 us more, and 16-byte loads across the ends of rows of no multiple of four columns 1.5.
//
// Measured, one handle launched again and again, the quad-union kernel and this one: 2847 x 1952 x 8, 61 % sparse, 14.3 and 7.8 us
// (17.5 MB of copy); 4096 x 2048 x 16, 50 %, 16.0 and 11.3; 317 x 930 x 11, 74 %, 7.0 and 5.0; 10 x 512 x 4, 80 %, 5.0 (row
// kernel) and 4.3 (on another card 4.5 and 3.8).  Error against 64 bits: 0.67 of the replaced kernels' on average over 120 launches.
//
// More columns, in slabs of 16 or 32: pays where a matrix is so small that the quad-union kernel's exchange of partial tiles and its
// tiles' barriers are most of the launch: 51 x 697 x 208, 58 % sparse, 7.0 and 5.4 us; 256 x 1136 x 36, 69 %, 7.6 and 5.8; 45 x 757 x 224, 75 %
// (shared gather) 6.1 and 5.4.  Every slab reads the copy of the matrix again, so large ones stay there.
//
// Sums, zero weights and values that are not finite: as there.  With an infinity in one column of X / in each, us: 2847 x 1952 x 8 16 / 21 (the quad-union
// kernel 35 / 52), 1067 x 900 x 28, 60 %, 11 / 27 (12 / 36), 256 x 1136 x 36 8 / 15 (10 / 28), 2000 x 1500 x 3, 50 %, 13 / 13 (row kernel 12); output
// by output, a whole wave for each, it took 24 / 90, 13 / 116, 10 / 80 and 18 / 42.
#include "so_internal.h"
#include "exact_outputs.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

constexpr uint32_t KT = so_quads::kTileRows, WAVES = 16, LOG_WAVES = 4, THREADS = WAVES * 64, AHEAD = 4;
constexpr uint32_t MOST_GROUPS = 10 * THREADS;   // 16-byte groups of X in LDS: 160 KB
constexpr uint32_t RED_BYTES = THREADS * 8;       // the waves' sums, in the place of X
constexpr uint32_t MOST_COLUMNS = 65535u * 16u;   // slabs of 16 are counted by blockIdx.y

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct NarrowArgs {
    const float *w;             // [chunks][64]
    const uint8_t *off;         // [chunks][16]: the X row inside its tile
    const uint2 *info;          // [quads][ntiles] {first chunk, units of four steps}
    uint32_t m, n, C, nquads, ntiles, qw_log2, magic;   // magic: e / C is the high half of e * magic (e < 2^19, 1 < C <= 32)
    const float *X, *bias;
    float *Y;
    const float *Wd;            // the ROW arrays, for outputs that are computed again
    const uint32_t *idx, *nnz;
    uint32_t r;
};

__device__ __forceinline__ float xor_add(float keep, float send, int mask) { return keep + __shfl_xor(send, mask, 64); }

// V values of a row of X per lane and LDS read, R reads per chunk: 4 V R columns.
template <int V, int R, int ACT>
__global__ __launch_bounds__(THREADS)
void ellpack_matmul_narrow_kernel(NarrowArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr uint32_t GROUPS = V * R;                               // 16-byte groups of an X row in LDS
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t qw = 1u << a.qw_log2, kw = WAVES >> a.qw_log2;
    const uint32_t wq = wave & (qw - 1u), wk = wave >> a.qw_log2, quad = (blockIdx.x << a.qw_log2) + wq;
    const uint32_t c0 = blockIdx.y * (4u * GROUPS), cols = min(a.C - c0, 4u * GROUPS);       // the slab's columns

    // the wave's chunks: every kw-th of the quad's.  Lane t holds the first chunk of tile t, so the tile of a chunk is a count of lanes.
    uint32_t first = 0xffffffffu, begin = 0, end = 0;
    if (quad < a.nquads) {
        const uint2 *inf = a.info + (size_t)quad * a.ntiles;
        if (lane < a.ntiles) first = inf[lane].x;
        const uint2 last = inf[a.ntiles - 1u];
        begin = __builtin_amdgcn_readfirstlane(inf[0].x) + wk;
        end = __builtin_amdgcn_readfirstlane(last.x + ((last.y + 3u) >> 2));
    }
    const uint32_t count = begin < end ? (end - begin + kw - 1u) >> (LOG_WAVES - a.qw_log2) : 0u;
    struct Batch { float w[AHEAD]; uint32_t o[AHEAD]; };
    auto request = [&](Batch &b, uint32_t i) {                       // past the last chunk: the last one again
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) {
            const size_t c = begin + min(i + u, count - 1u) * kw;
            b.w[u] = a.w[c * 64u + lane];
            if constexpr (R == 1) b.o[u] = a.off[c * 16u + (lane >> 2)];
            else b.o[u] = reinterpret_cast<const uint16_t *>(a.off)[c * 8u + (lane >> 3)];
        }
    };
    Batch b0, b1;
    if (count != 0u) { request(b0, 0u); request(b1, AHEAD); }

    // X into LDS, four values per thread and load, all loads in flight: as it lies in memory, and from there to the rows'
    // places, a value at a time where rows are no whole groups of four (128-bit loads across the rows' ends took 1.5 us longer).
    const uint32_t total = a.n * a.C, groups = (total + 3u) / 4u;
    auto stage = [&](auto loads) {
        constexpr uint32_t N = decltype(loads)::value;
        f32x4 v[N];
#pragma unroll
        for (uint32_t u = 0; u < N; ++u) v[u] = *reinterpret_cast<const f32x4u *>(a.X + min(4u * (tid + u * THREADS), total - 4u));
#pragma unroll
        for (uint32_t u = 0; u < N; ++u) {
            if (tid + u * THREADS >= groups) break;
            const uint32_t e = min(4u * (tid + u * THREADS), total - 4u);     // (the last group again covers part of the one before)
            uint32_t row = a.C == 1u ? e : __umulhi(e, a.magic), col = e - row * a.C;
            if (a.C % 4u == 0u) {
                *reinterpret_cast<f32x4 *>(lds + row * (GROUPS * 16u) + col * 4u) = v[u];
                continue;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                *reinterpret_cast<float *>(lds + row * (GROUPS * 16u) + col * 4u) = v[u][k];
                if (++col == a.C) { col = 0u; ++row; }
            }
        }
    };
    // Slabs: C is a multiple of four.  Places past the last column get values of others, which reach no output.
    auto stage_slab = [&](auto loads) {
        constexpr uint32_t N = decltype(loads)::value;
        const float *const X = a.X + c0;
        f32x4 v[N];
#pragma unroll
        for (uint32_t u = 0; u < N; ++u) {
            const uint32_t g = min(tid + u * THREADS, a.n * GROUPS - 1u);
            v[u] = *reinterpret_cast<const f32x4u *>(X + ((size_t)(g / GROUPS) * a.C + min(g % GROUPS * 4u, cols - 4u)));
        }
#pragma unroll
        for (uint32_t u = 0; u < N; ++u)
            if (tid + u * THREADS < a.n * GROUPS) reinterpret_cast<f32x4 *>(lds)[tid + u * THREADS] = v[u];
    };
    if (gridDim.y > 1u) {
        if constexpr (GROUPS >= 4u) {
            if (a.n * GROUPS <= 4u * THREADS) stage_slab(std::integral_constant<uint32_t, 4>());
            else stage_slab(std::integral_constant<uint32_t, MOST_GROUPS / THREADS>());
        }
    } else if (total < 4u) {
        if (tid < total) *reinterpret_cast<float *>(lds + tid / a.C * (GROUPS * 16u) + tid % a.C * 4u) = a.X[tid];
    } else if (groups <= 4u * THREADS) stage(std::integral_constant<uint32_t, 4>());
    else stage(std::integral_constant<uint32_t, MOST_GROUPS / THREADS>());
    __syncthreads();

    // Four accumulators at least: a chain of multiply-adds takes every SETS-th chunk, which rounds less and waits less.
    constexpr int SETS = 4 / V;
    f32x4 part[SETS][V];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int v = 0; v < V; ++v) part[i][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    const char *const mine = lds + (lane % (4u * R)) * (V * 4u);
    auto multiply = [&](const Batch &b, uint32_t i) {
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) {
            const uint32_t c = begin + min(i + u, count - 1u) * kw;
            const uint32_t tile = (uint32_t)__popcll(__ballot(first <= c)) - 1u;
            const float w = i + u < count ? b.w[u] : 0.0f;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t row = tile * KT + (R == 1 ? b.o[u] : (b.o[u] >> (8 * k)) & 255u);
                const float *x = reinterpret_cast<const float *>(mine + row * (GROUPS * 16u));
                float xv[V];
                if constexpr (V == 4) { const f32x4 t = *reinterpret_cast<const f32x4 *>(x); xv[0] = t[0]; xv[1] = t[1]; xv[2] = t[2]; xv[3] = t[3]; }
                else if constexpr (V == 2) { const float2 t = *reinterpret_cast<const float2 *>(x); xv[0] = t.x; xv[1] = t.y; }
                else xv[0] = x[0];
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    f32x4 *const acc = part[u % SETS];
                    if constexpr (R == 1) acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, xv[v], acc[v], 0, 0, 0);
                    else if (k == 0) acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, xv[v], acc[v], 1, 0, 0);
                    else acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, xv[v], acc[v], 1, 1, 0);
                }
            }
        }
    };
    for (uint32_t i = 0; i < count; i += 2u * AHEAD) {
        multiply(b0, i);
        request(b0, i + 2u * AHEAD);
        if (i + AHEAD >= count) break;
        multiply(b1, i + AHEAD);
        request(b1, i + 3u * AHEAD);
    }

    f32x4 acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = SETS == 4 ? (part[0][v] + part[1 % SETS][v]) + (part[2 % SETS][v] + part[3 % SETS][v]) : SETS == 2 ? part[0][v] + part[1 % SETS][v] : part[0][v];
    // Sum over the groups of lanes, halving what a lane holds: row lane / 16 of the quad after two exchanges, then columns.
    float s[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const u32x2 p = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[v][0]), __float_as_uint(acc[v][2]), false, false);
        const u32x2 q = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[v][1]), __float_as_uint(acc[v][3]), false, false);
        const float s02 = __uint_as_float(p[0]) + __uint_as_float(p[1]), s13 = __uint_as_float(q[0]) + __uint_as_float(q[1]);
        const u32x2 e = __builtin_amdgcn_permlane16_swap(__float_as_uint(s02), __float_as_uint(s13), false, false);
        s[v] = __uint_as_float(e[0]) + __uint_as_float(e[1]);
    }
    const bool hi8 = lane & 8u, hi4 = lane & 4u;
    float out[R];
    uint32_t col;
    if constexpr (R == 2) {
        out[0] = xor_add(hi8 ? s[2] : s[0], hi8 ? s[0] : s[2], 8);
        out[1] = xor_add(hi8 ? s[3] : s[1], hi8 ? s[1] : s[3], 8);
        col = (lane & 7u) * 4u + (hi8 ? 2u : 0u);
    } else if constexpr (V == 4) {
        const float t0 = xor_add(hi8 ? s[2] : s[0], hi8 ? s[0] : s[2], 8), t1 = xor_add(hi8 ? s[3] : s[1], hi8 ? s[1] : s[3], 8);
        out[0] = xor_add(hi4 ? t1 : t0, hi4 ? t0 : t1, 4);
        col = (lane & 3u) * 4u + (hi8 ? 2u : 0u) + (hi4 ? 1u : 0u);
    } else if constexpr (V == 2) {
        const float t = xor_add(hi8 ? s[1] : s[0], hi8 ? s[0] : s[1], 8);
        out[0] = xor_add(t, t, 4);
        col = hi4 ? 0xffffu : (lane & 3u) * 2u + (hi8 ? 1u : 0u);    // (lanes with bit 2 hold the same again)
    } else {
        const float t = xor_add(s[0], s[0], 8);
        out[0] = xor_add(t, t, 4);
        col = hi4 || hi8 ? 0xffffu : lane & 3u;
    }
    // Sum over the waves of a quad, through LDS.
    if (kw > 1u) {
        float *red = reinterpret_cast<float *>(lds);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k) red[(wave * R + k) * 64u + lane] = out[k];
        __syncthreads();
        if (wk == 0) {                                               // pairwise: a third less rounding than one after the other
#pragma unroll
            for (int k = 0; k < R; ++k) {
                float t[WAVES];
#pragma unroll
                for (uint32_t i = 0; i < WAVES; ++i) t[i] = i < kw ? red[(((i << a.qw_log2) + wq) * R + k) * 64u + lane] : 0.0f;
#pragma unroll
                for (uint32_t step = 1; step < WAVES; step *= 2)
#pragma unroll
                    for (uint32_t i = 0; i < WAVES; i += 2u * step) t[i] += t[i + step];
                out[k] = t[0];
            }
        }
    }
    if (wk != 0 || quad >= a.nquads) return;
    const uint32_t row = quad * 4u + (lane >> 4);
    const auto live = [&](int k) { return row < a.m && col + k < cols; };
    // A zero weight times a value of X that is not finite: outputs that came out as NaN are computed again from the
    // rows' own nonzeros, a group of four columns of all four rows at a time.
    uint32_t lost = 0;                                               // a bit per group
#pragma unroll
    for (int k = 0; k < R; ++k) lost |= live(k) && __builtin_isnan(out[k]) ? 1u << (col >> 2) : 0u;
    if (__builtin_expect(__ballot(lost != 0u) != 0u, 0)) {
#pragma unroll 1
        for (uint32_t g = 0; g < GROUPS; ++g) {
            if (__ballot(lost >> g & 1u) == 0u) continue;
            const uint32_t at = c0 + g * 4u, first = min(at, max(a.C, 4u) - 4u);               // four columns that exist, or all there are
            const so_f32x4 e = a.C >= 4u ? exact_outputs(a, row, first, lane & 15u) : exact_outputs<false>(a, row, first, lane & 15u);
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t v = c0 + col + k - first;
                const float again = v == 0u ? e[0] : v == 1u ? e[1] : v == 2u ? e[2] : e[3];
                if (col >> 2 == g && live(k) && __builtin_isnan(out[k])) out[k] = again;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
        if (live(k)) a.Y[(size_t)row * a.C + c0 + col + k] = so_epilogue<ACT>(out[k] + (a.bias ? a.bias[row] : 0.0f));
}

// 16-byte groups of a row of X in LDS for C <= 32 columns.
uint32_t groups_for(uint32_t C) { return C <= 4 ? 1u : C <= 8 ? 2u : C <= 16 ? 4u : 8u; }

template <int V, int R>
so_status launch(so_ctx *ctx, const NarrowArgs &a, dim3 blocks, size_t lds, int act)
{
#define SO_NARROW(A)                                                                              \
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_matmul_narrow_kernel<V, R, A>));           \
    ellpack_matmul_narrow_kernel<V, R, A><<<blocks, THREADS, lds, ctx->stream>>>(a);              \
    break
    switch (act) {
    case SO_ACT_RELU:    SO_NARROW(SO_ACT_RELU);
    case SO_ACT_SIGMOID: SO_NARROW(SO_ACT_SIGMOID);
    case SO_ACT_TANH:    SO_NARROW(SO_ACT_TANH);
    default:             SO_NARROW(SO_ACT_NONE);
    }
#undef SO_NARROW
    return SO_OK;
}

size_t lds_bytes(uint32_t n, uint32_t groups) { return std::max<size_t>((size_t)n * groups * 16u, RED_BYTES); }

bool fits(const so_ctx *ctx, const so_ellpack *E, uint32_t groups)
{
    return (uint64_t)E->n * groups <= MOST_GROUPS && lds_bytes(E->n, groups) <= (size_t)ctx->max_lds_bytes;
}

} // namespace

bool so_matmul_narrow_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return E->quads.d_w != nullptr && E->n != 0 && C >= 1 && C <= MOST_COLUMNS && (C <= 32 || C % 4 == 0) && E->quads.ntiles <= 64 && fits(ctx, E, C <= 32 ? groups_for(C) : 4u);
}

// Up to 32 columns the narrowest slab that holds them, beyond (whole groups of four only: the others' copies take up to twice as
// long) slabs of 16 or 32 columns (blockIdx.y), whichever is estimated faster; as few quads per workgroup as give no more workgroups than compute units.  The estimate -- the launch, a workgroup's
// start and its copy of X, the chunks of a wave, the bytes that slabs share -- was fitted to 696 launches of 10..4096 rows, 512..4096 columns, 1..64 dense
// columns, 50-95 % sparse on three cards, one handle again and again: 0.7 % too low on average, 5 % off (standard deviation; the same handle differs by
// as much from one allocation to the next), 20 % at most.  Slabs also to 320 launches of up to 1500 rows and 4800 dense columns, 10 % off: once X is more than an XCD's
// 4 MB of L2, the 64 bytes of a row that a slab of 16 takes cost a whole line from beyond it (4 x 1792 x 3780, 27 MB, 14.2 us, shared gather
// 7.6; 12 x 2172 x 1860 17.7, quad-union 8.5); those of 32 columns take whole lines.
so_narrow_plan so_matmul_narrow_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    const so_quads &Q = E->quads;
    so_narrow_plan best{};
    best.us = 1e30;
    for (uint32_t groups : {1u, 2u, 4u, 8u}) {
        if (C <= 32 ? groups != groups_for(C) : groups < 4u || !fits(ctx, E, groups)) continue;
        const uint32_t slabs = so_ceil_div(C, 4u * groups);
        uint32_t ql = 0;
        while (ql < LOG_WAVES && (uint64_t)so_ceil_div(Q.nquads, 1u << ql) * slabs > (uint64_t)ctx->compute_units) ++ql;
        const double rounds = so_ceil_div((uint64_t)so_ceil_div(Q.nquads, 1u << ql) * slabs, (uint64_t)ctx->compute_units);
        const double copy = 1e-4 * E->n * (slabs > 1 ? 4.6 * groups : C) * (C % 4u ? 0.6 : 0.45), chunks = (double)Q.total_chunks / Q.nquads * (1u << ql) / WAVES;
        const double megabytes = 4.0 * E->n * C / (1u << 20), far = slabs > 1 && groups == 4u && megabytes > 4.0 ? 0.6 * megabytes : 0.0;
        const double us = 3.0 + rounds * (1.0 + (slabs > 1 ? 0.2 : 0.0) + (groups == 8u ? 0.55 : 0.0) + copy + chunks * (0.077 + 0.021 * groups)) + 0.84e-5 * Q.total_chunks + far;
        if (us < best.us) best = so_narrow_plan{ql, groups, slabs, us};
    }
    return best;
}

so_status so_matmul_narrow_launch(so_ctx *ctx, const so_ellpack *E, const so_narrow_plan &p, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    const so_quads &Q = E->quads;
    const NarrowArgs a{Q.d_w, (const uint8_t *)Q.d_off, Q.d_info, E->m, E->n, C, Q.nquads, Q.ntiles, p.qw_log2, (uint32_t)(((1ull << 32) + C - 1u) / C),
                       dX, dBias, dY, E->d_Wd, E->d_idx, E->d_nnz, E->r};
    const dim3 blocks(so_ceil_div(Q.nquads, 1u << p.qw_log2), p.slabs);
    const size_t lds = lds_bytes(E->n, p.groups);
    switch (p.groups) {
    case 1:  return launch<1, 1>(ctx, a, blocks, lds, act);
    case 2:  return launch<2, 1>(ctx, a, blocks, lds, act);
    case 4:  return launch<4, 1>(ctx, a, blocks, lds, act);
    default: return launch<4, 2>(ctx, a, blocks, lds, act);
    }
}
