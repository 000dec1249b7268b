// The device encoder from one read of W: so_ellpack_encode_noalloc where the caller waits for the counts.
//
// ELLPACK's row pitch is the longest row's length, which is known only when every row has been looked at, so the two
// passes of csrc/runtime.hip read W twice.  Here one workgroup per compute unit takes its rows piece by piece, keeps what
// it finds -- values, a byte of column each -- in the 160 KB of its compute unit's LDS (40 MB over the chip), tells the
// others its longest row and its count, waits for theirs and writes its rows out at the pitch they agree on.  Pieces
// that LDS has no room for are read and packed again.
//
// Decomposition.  A piece is up to 2048 columns of a row (less where a workgroup would have fewer pieces than waves); the
// 16 waves take a workgroup's pieces in turn, each the next one's eight 16-byte loads ahead of the one it packs.  A wave packs into a
// part of LDS of its own, from the front on: nothing is synchronised until all pieces are counted.  A row's places are
// then a prefix sum over its pieces.
//
// The wait for the other workgroups has every one of them resident (a workgroup per compute unit), unless somebody else's
// kernel holds some of the chip: it gives up after a bounded number of looks, the host is told, and the two passes do
// the call again, and the context's next ones.  The words the workgroups tell each other carry the call's number, so nothing needs clearing.  One
// wave of each looks, at four workgroups per lane, and everything it adds up is in DPP steps: the places, the wait and the agreement took 1.2, 3.0 and 1.0 us by
// barriers and shuffles over the workgroup, and 0.6, 1.8 and 0.2 now.
//
// Results of up to kThroughSlots slots are stored past the L2, and the first workgroup tells the host when all are done: the end of the kernel, its
// writing back of the caches, and a kernel or a wait of the runtime's behind it cost 3 us more.
//
// What bounds it: the read of W (8192 x 8192: 42 to 63 us, by workgroup and XCD, half of them at 50; the copy's rate would take 43), then what
// follows the slowest workgroup: 1.5 us until all know of all, 12 to 14 of writing 61 MB at 90 % sparse; launch and the host's
// wait 14, its word 10 (clock stamps).  Memory moves 269 MB in, W once, and 61 out (counters); at 50 % sparse, where LDS keeps one piece of eight, 450 in.
// The whole call on one matrix again and again, two passes / this one with the host told behind the kernel / this one, us:
//
//   8192 x 8192 at 97 / 50 % sparse                            100 / 78.9 / 74.2, 195 / 174 / 174
//   4096 x 4096, 2199 x 2165 at 90 %, 5442 x 2598 at 63 %      45 / 33.4 / 30.5,  27 / 22.9 / 20.8,  - / 39.6 / 37.1
//   8192 x 8192 at 97 / 90 %, 2199 x 2165 at 91 %, changing matrices   - / 85.9 / 80.3, 127.6 / 92.9 / 91.6,  - / 24.7 / 22.8
#include "so_internal.h"

#include <atomic>
#include <type_traits>

namespace {

constexpr uint32_t THREADS = 1024, WAVES = 16, GROUPS = 8;        // groups of 256 columns a piece has at most
constexpr uint32_t HEAD = 256;                                    // bytes of LDS before the table of counts
constexpr uint32_t kEntryLimit = 4096;                            // words of the table of counts
constexpr uint32_t MOST_WGS = 256, kGaveUp = 0xffffffffu;
// Up to this many slots of the result are stored past the L2, and the host is told from the kernel; beyond, the caches' writing together of neighbouring pieces gains
// more than the end of the kernel and its wait cost.  Changing matrices, slots, us past the L2 / not: 4096 x 4096 at 80 % sparse, 3.5 M, 39.2 / 41.3, 5442 x 2598 at 63 %, 5.3 M,
// 45.5 / 47.1, 3491 x 4690 at 56 %, 7.5 M, 52.4 / 49.2, 8192 x 8192 at 97 / 90 %, 2.2 and 7.5 M, 80.3 / 84.6, 99 to 109 / 91.6.
constexpr uint64_t kThroughSlots = 6u << 20;
static_assert(3 * MOST_WGS <= 2 * kEncodeTold, "the words have room");
// Of a bounded wait, 0.19 us each: 3 ms.  The workgroups end the read of 8192 x 8192 some 16 to 21 us apart, of 32768 x 32768 115; those of a result that is stored past the L2 are
// done 2 to 4 us apart.  The rest is for whoever holds part of the chip for a while: giving up costs this call the two passes and the next ones too.
constexpr uint32_t kLooks = 1u << 14;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Where one pass is the faster: the workgroups' wait for one another costs 3 us more than a second launch, which a matrix of
// 16 MB repays (us, two passes / one: 256 x 8192 20.1 / 24.4, 911 x 1901 23.6 / 25.4, 1289 x 6285 30.7 / 28.4, 2048 x 2048 26.8 / 24.1); rows
// well below three groups of 256 columns leave lanes idle (16384 x 520 35.5 / 40.2, 40000 x 600 60.2 / 69.4, 6549 x 786 35.3 / 31.3); and few
// rows divide badly over the workgroups (520 rows, three on some, two on most: 22.5 / 24.2; 512 rows 30.5 / 27.4).
//
// No upper size: beyond what LDS holds (6.7 M nonzeros) the gain goes, but little is lost.  Us, two passes / one: 16384 x 16384 with 5 / 10 / 50 % kept
// 418 / 350, 454 / 438, 664 / 675; 32768 x 16384 with 2 / 10 / 50 % 769 / 605, 880 / 910, 1287 / 1336; 32768 x 32768 1518 / 1427, 1811 / 1838, 2489 / 2359;
// few long rows gain most (256 x 100 000 at 10 % 64 / 42, 4 x 2 000 000 685 / 348).  Not settled: rows whose last group is mostly empty, at few
// nonzeros, 50 001 x 800 with 5 / 10 / 50 % 74 / 83, 77 / 83, 128 / 109; 500 000 x 800 665 / 706, 747 / 836, 1220 / 1065: how many are kept is not known before.
constexpr uint64_t kLeastElements = 4u << 20;
constexpr uint32_t kLeastColumns = 768;

struct EncodeArgs {
    const float *W;
    uint32_t m, n, r_cap, groups, segs, part, table_bytes, call, looks;
    unsigned long long *told;        // [3][MOST_WGS]: {call, longest row}, {call, nonzeros}, {call, 0} when done
    uint32_t *host, *nnz, *idx;
    float *Wd;
    so_tell tell;
};

// THROUGH: stores past the L2, which other compute units and streams do not share: what has been written is there when the host is told, without the end of
// the kernel.  (The s_nop: a store of 16 bytes reads its registers late, which the compiler sees to for its own stores only.)
template <bool THROUGH, typename T>
__device__ __forceinline__ void store(T *p, T v)
{
    if constexpr (THROUGH) so_store_through(p, v);
    else *p = v;
}
template <bool THROUGH, typename T, typename V>
__device__ __forceinline__ void store4(T *p, V v)
{
    if constexpr (THROUGH) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
    else *reinterpret_cast<V *>(p) = v;
}

// Over the 64 lanes, in DPP steps; in every lane.
template <bool MAX>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v)
{
    const auto step = [&](uint32_t u) { v = MAX ? max(v, u) : v + u; };
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));      // row_shr:1, 2, 4, 8
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, true));      // row_bcast:15 into rows 1 and 3, :31 into 2 and 3
    step(__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, true));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// A packed piece of c entries: the counts after each group but the last (two bytes each), values, column bytes.
__device__ __forceinline__ uint32_t piece_bytes(uint32_t c) { return 16u + ((c * 5u + 15u) & ~15u); }

__device__ __forceinline__ uint32_t piece_count(const f32x4u (&v)[GROUPS])
{
    uint32_t c = 0;
#pragma unroll
    for (uint32_t u = 0; u < GROUPS; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) c += (uint32_t)__popcll(__ballot(v[u][e] != 0.0f));
    return c;
}

// Packs the piece a wave holds (a lane has four consecutive columns of each group) to `to` in ascending column order.
__device__ __forceinline__ void piece_pack(const f32x4u (&v)[GROUPS], uint32_t c, char *to, uint32_t lane)
{
    float *val = reinterpret_cast<float *>(to + 16);
    uint8_t *col = reinterpret_cast<uint8_t *>(to + 16u + 4u * c);
    uint32_t at = 0, ends[GROUPS / 2];
#pragma unroll
    for (uint32_t u = 0; u < GROUPS; ++u) {
        uint32_t pos = at;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint64_t mask = __ballot(v[u][e] != 0.0f);
            pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, pos));
            at += (uint32_t)__popcll(mask);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (v[u][e] != 0.0f) {
                val[pos] = v[u][e];
                col[pos] = (uint8_t)(lane * 4u + (uint32_t)e);
                ++pos;
            }
        if (u % 2u == 0u) ends[u / 2u] = at;
        else ends[u / 2u] |= at << 16;
    }
    if (lane == 0) *reinterpret_cast<uint4 *>(to) = make_uint4(ends[0], ends[1], ends[2], ends[3]);
}

// Writes a packed piece whose first column is c0 to the row's slots from wd, ix on, four entries per lane.
template <bool THROUGH>
__device__ __forceinline__ void piece_write(const char *from, uint32_t c, uint32_t c0, float *wd, uint32_t *ix, uint32_t lane)
{
    const float *val = reinterpret_cast<const float *>(from + 16);
    const uint8_t *col = reinterpret_cast<const uint8_t *>(from + 16u + 4u * c);
    const uint4 e4 = *reinterpret_cast<const uint4 *>(from);
    uint32_t ends[GROUPS];
    const uint32_t words[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
    for (uint32_t u = 0; u < GROUPS; ++u) ends[u] = __builtin_amdgcn_readfirstlane(u % 2u == 0u ? words[u / 2u] & 0xffffu : words[u / 2u] >> 16);
    auto column = [&](uint32_t k, uint32_t byte) {
        uint32_t g = 0;
#pragma unroll
        for (uint32_t u = 0; u + 1u < GROUPS; ++u) g += k >= ends[u] ? 256u : 0u;
        return c0 + g + byte;
    };
    for (uint32_t k = lane * 4u; k < c; k += 256u) {
        if (k + 4u <= c) {
            const uint32_t b = *reinterpret_cast<const uint32_t *>(col + k);
            store4<THROUGH>(wd + k, *reinterpret_cast<const f32x4u *>(val + k));
            store4<THROUGH>(ix + k, u32x4u{column(k, b & 0xffu), column(k + 1u, (b >> 8) & 0xffu), column(k + 2u, (b >> 16) & 0xffu), column(k + 3u, b >> 24)});
        } else {
            for (uint32_t i = k; i < c; ++i) {
                store<THROUGH>(wd + i, val[i]);
                store<THROUGH>(ix + i, column(i, col[i]));
            }
        }
    }
}

__global__ __launch_bounds__(THREADS)
void ellpack_encode_once_kernel(EncodeArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t *smax = reinterpret_cast<uint32_t *>(lds), *ssum = smax + WAVES, &agreed = smax[2 * WAVES];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wgs = gridDim.x, wg = blockIdx.x, rows = (a.m - wg + wgs - 1u) / wgs, items = rows * a.segs;     // rows wg, wg + wgs, ...
    uint32_t *table = reinterpret_cast<uint32_t *>(lds + HEAD);      // [rows][segs + 1]: counts, then the places of the pieces in their row
    char *part = lds + HEAD + a.table_bytes + wave * a.part;

    auto load = [&](uint32_t j, f32x4u (&v)[GROUPS]) {
        const uint32_t row = j / a.segs, c0 = (j - row * a.segs) * a.groups * 256u, jw = c0 + lane * 4u;
        const float *wr = a.W + (size_t)(wg + row * wgs) * a.n;
        if (a.groups == GROUPS && c0 + GROUPS * 256u <= a.n) {
#pragma unroll
            for (uint32_t u = 0; u < GROUPS; ++u) v[u] = *reinterpret_cast<const f32x4u *>(wr + jw + u * 256u);
        } else {
#pragma unroll
            for (uint32_t u = 0; u < GROUPS; ++u) {
                v[u] = f32x4u{0.f, 0.f, 0.f, 0.f};
                if (u >= a.groups) continue;
                const uint32_t c = jw + u * 256u;
                if (c + 4u <= a.n) v[u] = *reinterpret_cast<const f32x4u *>(wr + c);
                else {
                    if (c < a.n) v[u][0] = wr[c];
                    if (c + 1u < a.n) v[u][1] = wr[c + 1u];
                    if (c + 2u < a.n) v[u][2] = wr[c + 2u];
                }
            }
        }
    };

    // the pieces, counted, and packed while there is room
    f32x4u v[GROUPS], next[GROUPS];
    uint32_t used = 0;
    if (wave < items) load(wave, v);
    for (uint32_t j = wave; j < items; j += WAVES) {
        if (j + WAVES < items) load(j + WAVES, next);
        const uint32_t c = piece_count(v);
#pragma unroll
        for (uint32_t u = 0; u < GROUPS; ++u) asm volatile("" : "+v"(v[u]));     // the 32 ballots are taken again, not kept: they would not fit the scalar registers
        if (used + piece_bytes(c) <= a.part) {
            piece_pack(v, c, part + used, lane);
            used += piece_bytes(c);
        }
        if (lane == 0) table[j + j / a.segs] = c;
        if (j + WAVES < items) {
#pragma unroll
            for (uint32_t u = 0; u < GROUPS; ++u) v[u] = next[u];
        }
    }
    __syncthreads();

    // counts -> places; the workgroup's longest row and its count, by as many waves as 64 rows each take
    const uint32_t takers = min(WAVES, (rows + 63u) / 64u);
    if (wave < takers) {
        uint32_t vmax = 0, vsum = 0;
        for (uint32_t row = tid; row < rows; row += takers * 64u) {
            uint32_t *t = table + (size_t)row * (a.segs + 1u), at = 0;
            for (uint32_t s = 0; s < a.segs; ++s) { const uint32_t c = t[s]; t[s] = at; at += c; }
            t[a.segs] = at;
            so_store_through(a.nnz + wg + row * wgs, at);
            vmax = max(vmax, at);
            vsum += at;
        }
        vmax = wave_reduce<true>(vmax);
        vsum = wave_reduce<false>(vsum);
        if (lane == 0) { smax[wave] = vmax; ssum[wave] = vsum; }
    }
    if (takers > 1u) __syncthreads();
    // The first wave tells the other workgroups, and looks for their words, four per lane: word(value) for each that has come; true: all have.
    const auto put = [&](unsigned long long *words, uint32_t value) {
        __hip_atomic_store(words + wg, (unsigned long long)a.call << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const auto look_for_all = [&](const unsigned long long *words, auto &&start, auto &&word) {
        bool all = false;
        for (uint32_t look = 0; look < a.looks && !all; ++look) {
            unsigned long long x[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) x[i] = __hip_atomic_load(words + min(lane + 64u * i, wgs - 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool got = true;
            start();
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                got &= (uint32_t)(x[i] >> 32) == a.call;
                if (lane + 64u * i < wgs) word((uint32_t)x[i]);
            }
            all = __all(got);
            if (!all) __builtin_amdgcn_s_sleep(1);
        }
        return all;
    };
    const auto to_host = [&](uint32_t *word, uint32_t value) { __hip_atomic_store(word, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    if (wave == 0) {
        const uint32_t mine = wave_reduce<true>(lane < takers ? smax[lane] : 0u), sum = wave_reduce<false>(lane < takers ? ssum[lane] : 0u);
        if (lane == 0) { put(a.told, mine); put(a.told + MOST_WGS, sum); }
        uint32_t longest = 0;
        const bool all = look_for_all(a.told, [&]() { longest = 0; }, [&](uint32_t x) { longest = max(longest, x); });
        longest = wave_reduce<true>(longest);
        if (lane == 0) agreed = all ? longest : kGaveUp;
    }
    __syncthreads();
    const uint32_t r = __builtin_amdgcn_readfirstlane(agreed);
    const bool fits = r != kGaveUp && r <= a.r_cap, plain = fits && (uint64_t)a.m * r > kThroughSlots;
    // By the first workgroup's first wave: the longest row and all counts, or that somebody has given up, and the word that the host polls.
    const auto tell = [&]() {
        uint32_t low = 0, high = 0;
        const bool all = r != kGaveUp && look_for_all(a.told + MOST_WGS, [&]() { low = high = 0; }, [&](uint32_t x) { low += x & 0xffffu; high += x >> 16; });
        const unsigned long long total = ((unsigned long long)wave_reduce<false>(high) << 16) + wave_reduce<false>(low);
        if (lane == 0) {
            if (!all) to_host(a.host + 3, 1u);
            else { to_host(a.host, r); to_host(a.host + 1, (uint32_t)total); to_host(a.host + 2, (uint32_t)(total >> 32)); }
            if (plain) to_host(a.tell.flag + 2, 1u);
        }
        so_tell_now(a.tell);
    };
    if (r == kGaveUp && tid == 0) to_host(a.host + 3, 1u);
    if (plain && wg == 0 && wave == 0) tell();                    // from here on the host waits for the stream's end
    auto write_out = [&](auto through) {
        constexpr bool THROUGH = decltype(through)::value;
        // out: first the pieces that were kept, then the others, packed again now that LDS has room
        bool again = false;
        for (uint32_t pass = 0; pass == 0u || (pass == 1u && again); ++pass) {
            uint32_t at = 0;
            for (uint32_t j = wave; j < items; j += WAVES) {
                const uint32_t row = j / a.segs, s = j - row * a.segs;
                const uint32_t *t = table + (size_t)row * (a.segs + 1u) + s;
                const uint32_t first = __builtin_amdgcn_readfirstlane(t[0]), c = __builtin_amdgcn_readfirstlane(t[1]) - first, c0 = s * a.groups * 256u;
                const size_t slot = (size_t)(wg + row * wgs) * r + first;
                float *wd = a.Wd + slot;
                uint32_t *ix = a.idx + slot;
                const char *from = part + at;
                const bool kept = at + piece_bytes(c) <= a.part;
                if (kept) at += piece_bytes(c);
                else again = true;
                if (kept != (pass == 0u)) continue;
                if (pass == 0u) {
                    piece_write<THROUGH>(from, c, c0, wd, ix, lane);
                    continue;
                }
                if (j + WAVES < items) load(j, next);
                else {
#pragma unroll
                    for (uint32_t u = 0; u < GROUPS; ++u) next[u] = v[u];          // the wave's last piece is still here
                }
                if (piece_bytes(c) <= a.part) {
                    piece_pack(next, c, part, lane);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    piece_write<THROUGH>(part, c, c0, wd, ix, lane);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    continue;
                }
                uint32_t k = 0;                                       // more than a wave's part of LDS holds: straight to memory
#pragma unroll
                for (uint32_t u = 0; u < GROUPS; ++u) {
                    uint32_t pos = k;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint64_t mask = __ballot(next[u][e] != 0.0f);
                        pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, pos));
                        k += (uint32_t)__popcll(mask);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (next[u][e] != 0.0f) {
                            store<THROUGH>(wd + pos, (float)next[u][e]);
                            store<THROUGH>(ix + pos, c0 + u * 256u + lane * 4u + (uint32_t)e);
                            ++pos;
                        }
                }
            }
        }
        for (uint32_t row = wave; row < rows; row += WAVES) {
            const size_t slot = (size_t)(wg + row * wgs) * r;
            for (uint32_t k = table[(size_t)row * (a.segs + 1u) + a.segs] + lane; k < r; k += 64u) { store<THROUGH>(a.Wd + slot + k, 0.0f); store<THROUGH>(a.idx + slot + k, 0u); }
        }
        };
    if (plain) {
        write_out(std::false_type());
        return;
    }
    if (fits) write_out(std::true_type());
    // This workgroup is done; the first one tells the host when all are.
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");           // this wave's stores have arrived
    __syncthreads();
    if (wave != 0) return;
    if (lane == 0) put(a.told + 2u * MOST_WGS, 0u);
    if (wg != 0) return;
    const bool all = look_for_all(a.told + 2u * MOST_WGS, []() {}, [](uint32_t) {});
    if (!all && lane == 0) to_host(a.host + 3, 1u);
    tell();
}

} // namespace

so_status so_encode_once(so_ctx *ctx, const float *dDense, uint32_t m, uint32_t n, uint32_t r_cap, uint32_t *dNnz, float *dWd, uint32_t *dIdx,
                         void *told, uint32_t *host_header, bool *done, volatile uint32_t **at_end)
{
    *done = false;
    if ((uint64_t)m * n < kLeastElements || n < kLeastColumns) return SO_OK;
    const uint32_t wgs = std::min({m, (uint32_t)ctx->compute_units, MOST_WGS}), rows = so_ceil_div(m, wgs);
    if (4ull * m < 3ull * rows * wgs) return SO_OK;
    // pieces of equal width, one per wave at least
    const uint32_t n256 = so_ceil_div(n, 256u);
    uint32_t segs = std::max(so_ceil_div(n256, GROUPS), std::min(n256, so_ceil_div(WAVES, rows)));
    const uint32_t groups = so_ceil_div(n256, segs);
    segs = so_ceil_div(n256, groups);
    const uint64_t entries = (uint64_t)rows * (segs + 1u);
    if (entries > kEntryLimit) return SO_OK;
    const size_t lds = (size_t)ctx->max_lds_bytes;
    if (lds < (64u << 10)) return SO_OK;
    if (ctx->encode_spared != 0) {
        ctx->encode_spared -= std::min(ctx->encode_spared, (uint64_t)m * n);
        return SO_OK;
    }
    static std::atomic<uint32_t> calls{0};
    EncodeArgs a;
    a.W = dDense; a.m = m; a.n = n; a.r_cap = r_cap; a.groups = groups; a.segs = segs;
    a.table_bytes = ((uint32_t)entries * 4u + 15u) & ~15u;
    a.part = (uint32_t)((lds - HEAD - a.table_bytes) / WAVES) & ~15u;
    do a.call = ++calls; while (a.call == 0u);                    // zero is what the words held first
    a.looks = ctx->tune.wait_spins >= 0 ? (uint32_t)ctx->tune.wait_spins : kLooks;
    a.told = (unsigned long long *)told;
    a.host = host_header; a.nnz = dNnz; a.idx = dIdx; a.Wd = dWd;
    a.tell = so_tell_next(ctx);
    *at_end = a.tell.flag + 2;
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_encode_once_kernel));
    host_header[3] = a.tell.flag[2] = 0u;
    ellpack_encode_once_kernel<<<wgs, THREADS, lds, ctx->stream>>>(a);
    SO_LAUNCH_CHECK();
    ctx->last_kernel = "encode-once";
    *done = true;
    return SO_OK;
}
