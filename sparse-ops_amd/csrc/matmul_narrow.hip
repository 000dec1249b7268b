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
// chunks, which are requested four to eight ahead, the first before X.  No partial tiles are exchanged.
//
// What bounds it: small launches the latencies of launch (2.5 us) and first loads (1.1); in larger ones a chunk is 24 to 45 clocks of
// its compute unit, of which the MFMAs' 8 V R (at four columns a value and SIMD) and the copy's 288 bytes through L1 are about half each:
// without the MFMAs but one in four, the LDS reads or the requests 2048 x 2048 x 64 takes 8.3, 8.9 and 8.8 us of 9.8, with no loop 4.7.
// What it must not pay for is scalar instructions, which a SIMD issues at one in four clocks: with the tile of a chunk counted from
// a table, clamped requests and a select for the last ones there were 22 per chunk, and 97 clocks of the SIMD.  Hence whole row numbers
// (`rows`), fixed bases with one offset per batch, and a last batch of its own.  The LDS reads of a batch go out together, in front of its
// MFMAs.  Steps sorted so that a read's rows lie on different banks changed nothing.
//
// Measured, one handle launched again and again, the quad-union or column kernel, this one with scalar work per chunk and this one: 2847 x 1952 x 8, 61 % sparse,
// 11.5, 8.0 and 5.9 us (17.5 MB of copy); 4096 x 2048 x 16, 50 %, 15.2, 11.9 and 9.3; 317 x 930 x 11, 74 %, 5.6, 4.7 and 4.3; 139 x 1436 x 4,
// 60 %, 7.2, 4.7 and 3.7; 2048 x 2048 x 64, 80 %, 9.9, 12.7 and 9.6.  Error against 64 bits: 0.67
// of the replaced kernels' on average over 120 launches; the sums are the same bits in both forms of this one.
//
// More columns, in slabs of 16 or 32: pays where a matrix is so small that the quad-union kernel's exchange of partial tiles and its
// tiles' barriers are most of the launch: 51 x 697 x 208, 58 % sparse, 7.0 and 5.4 us; 256 x 1136 x 36, 69 %, 7.6 and 5.8; 45 x 757 x 224, 75 %
// (shared gather) 6.1 and 5.4 (with scalar work per chunk 4.7, 5.3 and 4.6 on another card, now 4.3, 5.2 and 4.3).  Every slab reads the copy of the matrix again, so large ones stay there.
//
// X a part at a time (PASSES), for any number of columns: what X in one piece is too large for, or too far from whole groups of four.  The quad-union kernel's
// launches of few rows and a long K are mostly its exchange of partial tiles; here a workgroup still has the whole of K and takes X in
// parts of 1280 rows (512 with slabs of 32 columns), two in LDS at a time, the first two asked for together.  A part costs 0.8 us beside its
// loads: the waves of a SIMD end a part at different times, by up to 1000 clocks, and all meet at its end (clock stamps).  Us, the other kernels / this
// one: quad-union 12 x 1238 x 173, 55 % sparse, 7.2 / 5.0, 125 x 1172 x 57, 54 %, 7.4 / 5.3, 84 x 692 x 149, 50 %, 7.0 / 5.2, 172 x 1992 x 29, 84 %, 7.6 / 6.3, 2000 x 2600 x 16, 60 %,
// 12.9 / 9.0; shared gather 26 x 745 x 91, 69 %, 5.9 / 4.9; column kernel 4022 x 1285 x 28, 59 %, 11.1 / 9.7; X in one piece 17 x 1090 x 28, 67 %, 6.0 / 4.7.
// From three parts on it gains little: 40 x 2835 x 83, 78 %, 7.9 / 7.7, 30 x 2988 x 56, 54 %, 7.3 / 7.6.
//
// Sums, zero weights and values that are not finite: as there.  With an infinity in one column of X / in each, us: 2847 x 1952 x 8 16 / 21 (the quad-union
// kernel 35 / 52), 1067 x 900 x 28, 60 %, 11 / 27 (12 / 36), 256 x 1136 x 36 8 / 15 (10 / 28), 2000 x 1500 x 3, 50 %, 13 / 13 (row kernel 12); output
// by output, a whole wave for each, it took 24 / 90, 13 / 116, 10 / 80 and 18 / 42.
#include "so_internal.h"
#include "lane_moves.h"
#include "exact_outputs.h"
#include "lds_sync.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

constexpr uint32_t WAVES = 16, LOG_WAVES = 4, THREADS = WAVES * 64, AHEAD = 4;
constexpr uint32_t MOST_GROUPS = 10 * THREADS;   // 16-byte groups of X in LDS: 160 KB
constexpr uint32_t RED_BYTES = THREADS * 8;       // the waves' sums, in the place of X
// Rows of X per pass, of which LDS holds two: whole tiles of the copy.  A pass's places in X are counted in 32 bits.
template <uint32_t GROUPS> constexpr uint32_t PASS_ROWS = GROUPS == 4u ? 1280u : 512u;
template <uint32_t GROUPS> constexpr uint32_t PASS_BYTES = PASS_ROWS<GROUPS> * GROUPS * 16u;
constexpr uint32_t MOST_PASS_COLUMNS = 65535u;
constexpr uint32_t MOST_COLUMNS = 65535u * 16u;   // slabs of 16 are counted by blockIdx.y
static_assert(2u * AHEAD * WAVES <= so_quads::kSlack && MOST_GROUPS <= so_quads::kMostRows, "what a wave requests is there");

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef const u32x2 __attribute__((address_space(4))) *const_info;

struct NarrowArgs {
    const float *w;             // [chunks][64]
    const uint16_t *rows;       // [chunks][16]: the X row
    const uint2 *info;          // [quads][ntiles] {first chunk, units of four steps}
    uint32_t m, n, C, nquads, ntiles, qw_log2, magic;   // magic: e / C is the high half of e * magic (e < 2^19, 1 < C <= 32)
    const float *X, *bias;
    float *Y;
    const float *Wd;            // the ROW arrays, for outputs that are computed again
    const uint32_t *idx, *nnz;
    uint32_t r;
};

// (By lane moves; through LDS a launch of 4.4 to 6 us takes 0.09 to 0.14 more.)
template <int D>
__device__ __forceinline__ float xor_add(float keep, float send) { return keep + so_lanes::across<D>(send); }

// V values of a row of X per lane and LDS read, R reads per chunk: 4 V R columns.  PASSES: X in LDS a part at a time.
template <int V, int R, int ACT, bool PASSES>
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

    // the wave's chunks: every kw-th of the quad's
    const uint32_t quarter = lane >> 2;
    uint32_t begin = 0, end = 0;
    if (quad < a.nquads) {
        const const_info inf = (const_info)(uintptr_t)(a.info + (size_t)quad * a.ntiles);
        const u32x2 first = inf[0], last = inf[a.ntiles - 1u];
        begin = first.x + wk;
        end = last.x + ((last.y + 3u) >> 2);
    }
    const uint32_t count = begin < end ? (end - begin + kw - 1u) >> (LOG_WAVES - a.qw_log2) : 0u;
    // Chunk i + u of a batch is at a base per u, which stays, and an offset for all of them, which moves: nothing scalar is issued per chunk.
    // Requests go up to two batches past the wave's last chunk, into other quads' chunks or the slack behind the last one (2 AHEAD WAVES chunks).
    const char *wb[AHEAD], *rb[AHEAD];
#pragma unroll
    for (uint32_t u = 0; u < AHEAD; ++u) {
        wb[u] = reinterpret_cast<const char *>(a.w) + (size_t)(begin + u * kw) * 256u;
        rb[u] = reinterpret_cast<const char *>(a.rows) + (size_t)(begin + u * kw) * 32u;
    }
    uint32_t wat = lane * 4u, rat = R == 1 ? quarter * 2u : (lane >> 3) * 4u;
    const uint32_t wstep = AHEAD * kw * 256u, rstep = AHEAD * kw * 32u;
    struct Batch { float w[AHEAD]; uint32_t row[AHEAD]; };
    auto request = [&](Batch &b) {
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) {
            b.w[u] = *reinterpret_cast<const float *>(wb[u] + wat);
            if constexpr (R == 1) b.row[u] = *reinterpret_cast<const uint16_t *>(rb[u] + rat);
            else b.row[u] = *reinterpret_cast<const uint32_t *>(rb[u] + rat);
        }
        wat += wstep;
        rat += rstep;
    };
    Batch b0, b1;
    // PASSES: the pass whose chunks are requested next, how many of them are not yet, and the wave's chunks of passes 0 .. `asking`.  Lane p holds
    // the wave's chunks of passes 0 .. p (a scalar load at the end of each pass would be waited for there).
    uint32_t asking = 0, unasked = 0, asked = 0, upto = 0;
    const uint32_t passes = (a.n + PASS_ROWS<GROUPS> - 1u) / PASS_ROWS<GROUPS>;      // 20 at most: 10 240 rows of 512
    if constexpr (PASSES) {
        const uint32_t t = (lane + 1u) * (PASS_ROWS<GROUPS> / so_quads::kTileRows);
        const uint32_t start = a.info[(size_t)min(quad, a.nquads - 1u) * a.ntiles + min(t, a.ntiles - 1u)].x, past = t < a.ntiles ? start : end;
        upto = past > begin && count != 0u ? (past - begin + kw - 1u) >> (LOG_WAVES - a.qw_log2) : 0u;
    }
    const auto chunks_up_to = [&](uint32_t pass) { return (uint32_t)__builtin_amdgcn_readlane(upto, pass); };
    // The next batch of the wave's: what is left of a pass where that is less than a batch, so that a batch never holds chunks of two passes.  The
    // marks keep its 2 AHEAD loads between them, and csrc/check_narrow_asks.py counts them there in the assembly of every build: `enter_pass` relies on it.
    auto ask = [&](Batch &b) {
        while (unasked == 0u && asking + 1u < passes) {
            const uint32_t all = chunks_up_to(++asking);
            unasked = all - asked;
            asked = all;
        }
        if (unasked == 0u) return 0u;
        asm volatile("; ask" : : : "memory");
        request(b);
        asm volatile("; asked" : : : "memory");
        const uint32_t some = min(unasked, AHEAD);
        unasked -= some;
        wat -= (AHEAD - some) * (wstep / AHEAD);
        rat -= (AHEAD - some) * (rstep / AHEAD);
        return 1u;
    };
    if constexpr (PASSES) {
        unasked = asked = chunks_up_to(0u);
        if (count != 0u) { (void)ask(b0); (void)ask(b1); }
    } else {
        if (count != 0u) { request(b0); request(b1); }
    }

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
    // PASSES: straight from memory into LDS, a pass in LOADS loads of 16 bytes per thread, into the two halves of LDS in turn; the first two passes
    // are asked for together.  Groups of four columns past the last column repeat the slab's first group and rows past the last row
    // repeat it (neither is ever used); a group that would end past the end of X (C not a multiple of 4, last row) is read from where
    // four values are left and shifted once it is in LDS.
    constexpr uint32_t ROWS = PASS_ROWS<GROUPS>, HALF = PASS_BYTES<GROUPS>, LOADS = (HALF + 16u * THREADS - 1u) / (16u * THREADS);
    const uint32_t sgrp = tid % GROUPS * 4u, srow = tid / GROUPS, xgrp = c0 + (sgrp < cols ? sgrp : 0u), lds0 = so_lds::lds_address(lds);
    const auto place = [&](uint32_t pass, uint32_t k) { return min(k * (THREADS / GROUPS) + srow, a.n - 1u - pass * ROWS) * a.C + xgrp; };
    const auto ends = [&](uint32_t pass) { return (uint32_t)min((uint64_t)(a.n - pass * ROWS) * a.C - 4u, (uint64_t)0x3ffffff0u); };   // the last place four values can be read from
    auto fetch_pass = [&](uint32_t pass) {
        const float *p = a.X + (size_t)pass * ROWS * a.C;
        const uint32_t to = lds0 + (pass & 1u) * HALF + wave * 1024u, e = ends(pass);
#pragma unroll
        for (uint32_t k = 0; k < LOADS; ++k)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         : : "v"(min(place(pass, k), e) * 4u), "s"(p), "s"(to + k * (16u * THREADS)) : "memory", "m0");
    };
    // This wave's part of a pass is in LDS, then everybody's; the next pass's way in.  Loads return in order: `asks` batches have been asked for
    // since the pass was, and may still be on their way.
    auto enter_pass = [&](uint32_t pass, uint32_t asks) {
        if (pass == 0u && passes > 1u) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LOADS) : "memory");      // pass 1 is on its way
        else if (asks >= 2u) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(4u * AHEAD) : "memory");
        else if (asks == 1u) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2u * AHEAD) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        if (a.C % 4u != 0u && pass + 1u == passes) {
            const uint32_t e = ends(pass);
#pragma unroll
            for (uint32_t k = 0; k < LOADS; ++k) {
                const uint32_t at = place(pass, k);
                if (at > e) {
                    f32x4 *q = reinterpret_cast<f32x4 *>(lds + (pass & 1u) * HALF + (k * THREADS + tid) * 16u);
                    const f32x4 u = *q;
                    const uint32_t shift = at - e;
                    *q = f32x4{shift == 1u ? u[1] : shift == 2u ? u[2] : u[3], shift == 1u ? u[2] : u[3], u[3], u[3]};
                }
            }
        }
        __syncthreads();
        if (pass != 0u && pass + 1u < passes) fetch_pass(pass + 1u);
    };
    if constexpr (PASSES) {
        fetch_pass(0u);
        if (passes > 1u) fetch_pass(1u);
        enter_pass(0u, 0u);
    } else if (gridDim.y > 1u) {
        if constexpr (GROUPS >= 4u) {
            if (a.n * GROUPS <= 4u * THREADS) stage_slab(std::integral_constant<uint32_t, 4>());
            else stage_slab(std::integral_constant<uint32_t, MOST_GROUPS / THREADS>());
        }
    } else if (total < 4u) {
        if (tid < total) *reinterpret_cast<float *>(lds + tid / a.C * (GROUPS * 16u) + tid % a.C * 4u) = a.X[tid];
    } else if (groups <= 4u * THREADS) stage(std::integral_constant<uint32_t, 4>());
    else stage(std::integral_constant<uint32_t, MOST_GROUPS / THREADS>());
    if constexpr (!PASSES) __syncthreads();

    // Four accumulators at least: a chain of multiply-adds takes every SETS-th chunk, which rounds less and waits less.
    constexpr int SETS = 4 / V;
    f32x4 part[SETS][V];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int v = 0; v < V; ++v) part[i][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t mine = lds0 + (lane % (4u * R)) * (V * 4u);       // of X's row 0, wherever the pass's first one lies
    typedef const __attribute__((address_space(3))) char *lds_pointer;
    struct Operands { float x[R][V]; };
    auto fetch = [&](uint32_t rows, Operands &o) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t row = R == 1 ? rows : k == 0 ? rows & 0xffffu : rows >> 16;
            const lds_pointer x = (lds_pointer)(mine + row * (GROUPS * 16u));
            if constexpr (V == 4) { const f32x4 t = *(const __attribute__((address_space(3))) f32x4 *)x; o.x[k][0] = t[0]; o.x[k][1] = t[1]; o.x[k][2] = t[2]; o.x[k][3] = t[3]; }
            else if constexpr (V == 2) { const f32x2 t = *(const __attribute__((address_space(3))) f32x2 *)x; o.x[k][0] = t[0]; o.x[k][1] = t[1]; }
            else o.x[k][0] = *(const __attribute__((address_space(3))) float *)x;
        }
    };
    auto multiply = [&](float w, const Operands &o, uint32_t u) {
        f32x4 *const acc = part[u % SETS];
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if constexpr (R == 1) acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, o.x[k][v], acc[v], 0, 0, 0);
                else if (k == 0) acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, o.x[k][v], acc[v], 1, 0, 0);
                else acc[v] = __builtin_amdgcn_mfma_f32_4x4x1f32(w, o.x[k][v], acc[v], 1, 1, 0);
            }
    };
    // a batch: its LDS reads, then its multiply-adds (a read at a time in front of its own leaves the reads' latency to the other waves)
    auto batch = [&](const Batch &b) {
        Operands o[AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) fetch(b.row[u], o[u]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u) multiply(b.w[u], o[u], u);
    };
    auto rest = [&](const Batch &b, uint32_t chunks) {
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; ++u)
            if (u < chunks) {
                Operands o;
                fetch(b.row[u], o);
                multiply(b.w[u], o, u);
            }
    };
    if constexpr (PASSES) {
        uint32_t pass = 0, done = chunks_up_to(0u), left = done, asks = 0;
        // to the next pass that has chunks for the wave; all waves enter every pass.  False: none is left.
        auto next_pass = [&]() {
            while (left == 0u) {
                if (++pass == passes) return false;
                const uint32_t all = chunks_up_to(pass);
                left = all - done;
                done = all;
                enter_pass(pass, asks);
                asks = 0u;
                mine = lds0 + (pass & 1u) * HALF - pass * HALF + (lane % (4u * R)) * (V * 4u);
            }
            return true;
        };
        auto some = [&](Batch &b) {
            if (left >= AHEAD) { batch(b); left -= AHEAD; }
            else { rest(b, left); left = 0u; }
            asks += ask(b);
            return left != 0u || next_pass();
        };
        if (next_pass())
            while (some(b0) && some(b1)) {}
    } else {
        uint32_t left = count;
        for (; left >= 2u * AHEAD; left -= 2u * AHEAD) {
            batch(b0);
            request(b0);
            batch(b1);
            request(b1);
        }
        if (left >= AHEAD) {
            batch(b0);
            rest(b1, left - AHEAD);
        } else rest(b0, left);
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
        out[0] = xor_add<8>(hi8 ? s[2] : s[0], hi8 ? s[0] : s[2]);
        out[1] = xor_add<8>(hi8 ? s[3] : s[1], hi8 ? s[1] : s[3]);
        col = (lane & 7u) * 4u + (hi8 ? 2u : 0u);
    } else if constexpr (V == 4) {
        const float t0 = xor_add<8>(hi8 ? s[2] : s[0], hi8 ? s[0] : s[2]), t1 = xor_add<8>(hi8 ? s[3] : s[1], hi8 ? s[1] : s[3]);
        out[0] = xor_add<4>(hi4 ? t1 : t0, hi4 ? t0 : t1);
        col = (lane & 3u) * 4u + (hi8 ? 2u : 0u) + (hi4 ? 1u : 0u);
    } else if constexpr (V == 2) {
        const float t = xor_add<8>(hi8 ? s[1] : s[0], hi8 ? s[0] : s[1]);
        out[0] = xor_add<4>(t, t);
        col = hi4 ? 0xffffu : (lane & 3u) * 2u + (hi8 ? 1u : 0u);    // (lanes with bit 2 hold the same again)
    } else {
        const float t = xor_add<8>(s[0], s[0]);
        out[0] = xor_add<4>(t, t);
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

template <int V, int R, bool PASSES = false>
so_status launch(so_ctx *ctx, const NarrowArgs &a, dim3 blocks, size_t lds, int act)
{
#define SO_NARROW(A)                                                                              \
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_matmul_narrow_kernel<V, R, A, PASSES>));   \
    ellpack_matmul_narrow_kernel<V, R, A, PASSES><<<blocks, THREADS, lds, ctx->stream>>>(a);      \
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

// Beyond 4 MB of X, an XCD's L2, what a launch of slabs waits for X from further away, by the workgroups that take a slab each: they lie on different XCDs, and each of the first
// three fetches the slab for itself.  A slab of 16 columns uses 64 bytes of every line.  Us per MB of X, measured less estimated without it, 260 launches of 4..2000 rows, 257..8000
// dense columns: slabs of 16 0.27, 0.58 and 0.7 for one, two, and three workgroups and more, of 32 0.12, 0.34 and 0.5.  (Without it X in parts was taken for 4 x 1187 x 3347 at 82 %
// sparse, 15 MB, 9.6 us, shared gather 5.8, and 5 x 2003 x 1119 at 84 %, 8.5 MB, 11.6, quad-union 7.5; whole X in slabs of 32 for 9 x 956 x 2264 at 67 %, 8.3 MB, 10.4, quad-union 7.0.)
static double narrow_far(uint32_t n, uint32_t C, uint32_t groups, uint32_t workgroups)
{
    const double megabytes = 4.0 * n * C / (1u << 20);
    static constexpr double us[2][3] = {{0.3, 0.6, 0.7}, {0.15, 0.35, 0.5}};
    return megabytes > 4.0 ? megabytes * us[groups == 8u][std::min(workgroups, 3u) - 1u] : 0.0;
}

bool so_matmul_narrow_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return E->quads.d_rows != nullptr && E->n != 0 && C >= 1 && C <= MOST_COLUMNS && (C <= 32 || C % 4 == 0) && fits(ctx, E, C <= 32 ? groups_for(C) : 4u);
}

// Up to 32 columns the narrowest slab that holds them, beyond (whole groups of four only: the others' copies take up to twice as
// long) slabs of 16 or 32 columns (blockIdx.y), whichever is estimated faster; as few quads per workgroup as give no more workgroups than compute units.  The estimate -- the launch, a workgroup's
// start and its copy of X (a value at a time where rows are no whole groups of four), the chunks of a wave, the copy's bytes, again for every
// slab of 32 -- was fitted to 228 launches of 10..4096 rows, 512..4096 columns, 4..256 dense columns, 50-95 % sparse, and 14 of up to
// 40 000 rows, one handle again and again: 7 % off (standard deviation; the same handle differs by 5 from one allocation to the next),
// 30 % at most; beyond 4 MB of X narrow_far is added.
// (Slabs of 16 are charged as for two workgroups, whatever there are.)
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
        const double copy = 1e-4 * E->n * (slabs > 1 ? 1.92 * groups : C * (C % 4u ? 0.95 : 0.73)), chunks = (double)Q.total_chunks / Q.nquads * (1u << ql) / WAVES;
        const double far = slabs == 1 ? 0.0 : narrow_far(E->n, C, groups, groups == 4u ? 2u : so_ceil_div(Q.nquads, 1u << ql));
        const double again = groups == 8u ? slabs : 1.0;                  // slabs of 32 columns are few enough for their reads of the copy to count
        const double us = 1.05 + rounds * (2.0 + (slabs > 1 ? 0.36 : 0.0) + copy + chunks * (0.025 + 0.0244 * groups)) + 0.75e-5 * Q.total_chunks * again + far;
        if (us < best.us) best = so_narrow_plan{ql, groups, slabs, false, us};
    }
    return best;
}

bool so_matmul_slabs_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return E->quads.d_rows != nullptr && E->n != 0 && C >= 4 && C <= MOST_PASS_COLUMNS && 2u * PASS_BYTES<4> <= (size_t)ctx->max_lds_bytes;
}

// Slabs of 16 or of 32 columns, whichever is estimated faster.  Fitted to 400 launches of 10..4096 rows, 512..4096 columns, 4..256 dense columns, 50-95 % sparse:
// 5.5 % off (standard deviation), 28 % at most; beyond 4 MB of X narrow_far is added.
so_narrow_plan so_matmul_slabs_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    const so_quads &Q = E->quads;
    so_narrow_plan best{};
    best.us = 1e30;
    for (uint32_t groups : {4u, 8u}) {
        if (ctx->tune.matmul_slabs > 0 && groups != (ctx->tune.matmul_slabs == 8 ? 8u : 4u)) continue;
        const uint32_t slabs = so_ceil_div(C, 4u * groups);
        uint32_t ql = 0;
        while (ql < LOG_WAVES && (uint64_t)so_ceil_div(Q.nquads, 1u << ql) * slabs > (uint64_t)ctx->compute_units) ++ql;
        const double wgs = (double)so_ceil_div(Q.nquads, 1u << ql) * slabs, cus = ctx->compute_units, rounds = std::ceil(wgs / cus);
        const double passes = so_ceil_div(E->n, groups == 4u ? PASS_ROWS<4> : PASS_ROWS<8>), chunks = (double)Q.total_chunks / Q.nquads * (1u << ql) / WAVES;
        const double copy = (groups == 4u ? 0.53e-3 : 0.474e-3) * E->n * std::min(1.0, wgs / cus);
        const double far = narrow_far(E->n, C, groups, so_ceil_div(Q.nquads, 1u << ql));
        const double us = 1.0 + rounds * (3.43 + 0.966 * (passes - 1.0) + copy + chunks * (0.0635 + 0.0142 * groups)) + 0.2e-5 * Q.total_chunks * (groups == 8u ? slabs : 1.0);
        if (us + far < best.us) best = so_narrow_plan{ql, groups, slabs, true, us + far};
    }
    return best;
}

so_status so_matmul_narrow_launch(so_ctx *ctx, const so_ellpack *E, const so_narrow_plan &p, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    const so_quads &Q = E->quads;
    const NarrowArgs a{Q.d_w, Q.d_rows, Q.d_info, E->m, E->n, C, Q.nquads, Q.ntiles, p.qw_log2, (uint32_t)(((1ull << 32) + C - 1u) / C),
                       dX, dBias, dY, E->d_Wd, E->d_idx, E->d_nnz, E->r};
    const dim3 blocks(so_ceil_div(Q.nquads, 1u << p.qw_log2), p.slabs);
    if (p.passes) return p.groups == 4u ? launch<4, 1, true>(ctx, a, blocks, 2u * PASS_BYTES<4>, act) : launch<4, 2, true>(ctx, a, blocks, 2u * PASS_BYTES<8>, act);
    const size_t lds = lds_bytes(E->n, p.groups);
    switch (p.groups) {
    case 1:  return launch<1, 1>(ctx, a, blocks, lds, act);
    case 2:  return launch<2, 1>(ctx, a, blocks, lds, act);
    case 4:  return launch<4, 1>(ctx, a, blocks, lds, act);
    default: return launch<4, 2>(ctx, a, blocks, lds, act);
    }
}
