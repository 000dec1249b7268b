// so_conv2d for small batches, and for small images at batches of 8, 16 and 32: a wave owns one output channel and 64 output columns, a column being one
// (pixel, batch entry) pair.
//
// The LDS-windowed kernel (csrc/conv.hip) gives a lane four batch entries of a pixel, so a batch of one is carried as
// four and a 7 x 7 layer of 512 channels keeps half of the chip's 1024 SIMDs busy with a quarter of their lanes.  Here
// a lane is a column, whatever the batch: TH x TW output pixels x B entries on 64 lanes, one 4-byte LDS read and one
// multiply-add per stored nonzero.  An output's multiply-adds form one chain in slot order (bias first), as everywhere
// in this library's convolutions: same bits.
//
// Decomposition.  A workgroup of G (16, 8 or 4) waves takes G channels on one tile.  The tile's input window -- all
// input channels if 150 KB of LDS hold them, else a chunk at a time -- is copied to LDS with zeros outside the image; a
// channel's entries {weight, LDS offset of its tap} come 16 at a time in lanes (the same 16 in every row of 16), eight
// such groups ahead, each group's place asked for again when it is done, and are handed round by DPP: per entry one address add, one read, one multiply-add.  The reads run
// three quads of entries ahead of the multiply-adds.  Workgroups shrink to 8 or 4 waves where that spreads the launch
// over more compute units.
//
// What bounds it: what one wave alone on a SIMD issues, about 5.8 clocks an instruction -- 18 clocks an entry in a loop of nothing else.  With
// four groups of entries ahead, asked for together, the loop's end waited for memory and the entry took 23; with eight, a place
// at a time, the ResNet-18-shaped stack at batch 1 takes 216.7 us instead of 230.8, a 7 x 7 x 512 layer (chains of 922) 14.4 instead of 16.2, a
// 14 x 14 x 256 one 9.8 instead of 11.0.  Before the chain come 3.0 us in which 16 waves issue the window's 592 copies, 12 clocks each (beginning in
// another place in each workgroup: 1.5 us slower; 16 bytes a lane instead of 4, with the pads cleared afterwards: 217.7 us for the stack), 1 until
// all is there, 0.6 of arguments and places, and the launch.
#include "so_internal.h"
#include "conv_internal.h"
#include "dpp_steps.h"

#include <cmath>
#include <cstring>

namespace {

struct ColArgs {
    uint32_t TH, TW, tiles_x;
    uint32_t PE;                 // pixels of a window plane in LDS order (rows of IP pixels)
    uint32_t IP, PL;             // row pitch in pixels; floats per plane (PE * B)
    uint32_t cc, nch, G, waves;  // channels per chunk, chunks; computing waves (= channels) and waves of a workgroup
    uint32_t pitch;              // groups from one (channel, chunk) to the next; 0: first[] says where they begin
    uint32_t sth, stw, sbh, sbw; // window pixels per output pixel, input pixels per window pixel
    uint32_t mB, mIP, mPL, mTW, mTilesX;
};

using so_dpp::fma4;
using so_dpp::step4;

constexpr uint32_t kAhead = 8;   // groups of entries a wave has asked for

// step(0) .. step(left - 1), at most kAhead - 1 of them.
template <uint32_t I, class F>
__device__ __forceinline__ void rest(uint32_t left, F &&step)
{
    if constexpr (I + 1u < kAhead) {
        if (left > I) {
            step(I);
            rest<I + 1u>(left, step);
        }
    }
}

// One convolution's operands.
struct ColCall {
    const int2 *entries;
    const uint32_t *first_group;
    const float *bias;
    float *Y;
    ColArgs a;
    so_conv_geom g;
    uint32_t relu;               // kActNoneOrRelu
};

template <int ACT>
__device__ __forceinline__ void column_convolution(const int2 *__restrict__ entries, const uint32_t *__restrict__ first_group, const ColArgs &a, const so_conv_geom &g,
                                                   const float *__restrict__ X, uint32_t B, const float *__restrict__ bias,
                                                   const float *__restrict__ resid, float *__restrict__ Y, uint32_t tile, uint32_t block, bool relu)
{
    extern __shared__ __attribute__((aligned(16))) float window[];     // [cc + 1][PL]: the last plane all zeros (padding entries point there)
    const uint32_t tid = threadIdx.x, lane = tid & 63u, threads = a.waves * 64u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t co = block * a.G + wave;
    const bool computes = wave < a.G && co < g.Cout;                   // the other waves only help copying
    const uint32_t tile_y = window_div(tile, a.tiles_x, a.mTilesX);
    const uint32_t th0 = tile_y * a.TH, tw0 = (tile - tile_y * a.tiles_x) * a.TW;

    // The wave's entries, groups of 16 (the stream ends with kAhead padding groups).  At a pitch their place needs no look
    // into a table, whose round trip to memory -- nothing is cached when a kernel starts -- would come before theirs.
    const uint32_t run0 = (computes ? co : 0u) * a.nch;
    const uint32_t l16 = lane & 15u;
    int2 held[kAhead];
    uint32_t g0, g1;
    const so_constant<uint32_t> first = (so_constant<uint32_t>)(uintptr_t)first_group;
    auto first_entries = [&](uint32_t t) {
        if (a.pitch != 0u) {
            g0 = (run0 + t) * a.pitch;
            g1 = g0 + __builtin_amdgcn_readfirstlane(first[run0 + t]);
        } else {
            g0 = __builtin_amdgcn_readfirstlane(first[run0 + t]);
            g1 = __builtin_amdgcn_readfirstlane(first[run0 + t + 1u]);
        }
        if (!computes) g1 = g0;
#pragma unroll
        for (uint32_t i = 0; i < kAhead; ++i) held[i] = (entries + (size_t)g0 * 16u)[i * 16u + l16];
    };
    first_entries(0);

    // this lane's output column
    const uint32_t pix = window_div(lane, B, a.mB), b = lane - pix * B;
    const uint32_t ty = window_div(pix, a.TW, a.mTW), tx = pix - ty * a.TW;
    const bool live = computes && pix < a.TH * a.TW && th0 + ty < g.H_out && tw0 + tx < g.W_out;
    const uint32_t lane_off = live ? ((ty * a.sth * a.IP + tx * a.stw) * B + b) * 4u : 0u;
    float acc = bias && computes ? ((so_constant<float>)(uintptr_t)bias)[co] : 0.0f;

    for (uint32_t k = tid; k < a.PL; k += threads) window[a.cc * a.PL + k] = 0.0f;
    // Input channels [t * cc, t * cc + cc) of the window, straight from memory into LDS: consecutive threads take
    // consecutive places -- of several planes at once where a plane is shorter than the workgroup -- and step over
    // channels; places outside the image are written with zeros instead.
    const bool several = a.PL < threads;
    const uint32_t per_pass = several ? window_div(threads, a.PL, a.mPL) : 1u;
    const uint32_t plane = several ? window_div(tid, a.PL, a.mPL) : 0u;
    const uint32_t image = g.H_in * g.W_in * B;
    const uint32_t lds0 = so_lds::lds_address(window) + wave * 256u;
    auto copy_window = [&](uint32_t t) {
        const uint32_t c0 = t * a.cc, cn = min(a.cc, g.Cin - c0);
        if (plane >= per_pass) return;
        uint32_t to = lds0;
        for (uint32_t e = tid - plane * a.PL; e < a.PL; e += threads, to += threads * 4u) {
            const uint32_t pe = window_div(e, B, a.mB), be = e - pe * B;
            const uint32_t ih = window_div(pe, a.IP, a.mIP), iw = pe - ih * a.IP;
            const int32_t gh = (int32_t)(th0 * g.stride_h + ih * a.sbh) - (int32_t)g.pad_h;
            const int32_t gw = (int32_t)(tw0 * g.stride_w + iw * a.sbw) - (int32_t)g.pad_w;
            if ((uint32_t)gh < g.H_in && (uint32_t)gw < g.W_in) {
                const uint32_t from = (plane * image + ((uint32_t)gh * g.W_in + (uint32_t)gw) * B + be) * 4u;
                const float *src = X + (size_t)c0 * image;
                // the last pass may hold fewer planes than this thread's
                const uint32_t whole = cn / per_pass * per_pass;
                uint32_t m0 = to;
                for (uint32_t c = 0; c < whole; c += per_pass) {
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(m0), "v"(from), "s"(src) : "memory", "m0");
                    src += (size_t)per_pass * image;
                    m0 += per_pass * a.PL * 4u;
                }
                if (whole + plane < cn)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(m0), "v"(from), "s"(src) : "memory", "m0");
            } else {
                for (uint32_t c = plane; c < cn; c += per_pass) window[c * a.PL + e] = 0.0f;
            }
        }
    };
    const uint32_t base = so_lds::lds_address(window) + lane_off;
    // Quads 1, 2 and 3 of the group before this one still owe their multiply-adds: operands in xB, xC, xD, weights in owed.
    float xA[4], xB[4] = {0.f, 0.f, 0.f, 0.f}, xC[4] = {0.f, 0.f, 0.f, 0.f}, xD[4] = {0.f, 0.f, 0.f, 0.f}, owed = -0.0f;
    auto group = [&](const int2 &e) {
        float w = __int_as_float(e.x);
        uint32_t off = (uint32_t)e.y;
        asm volatile("s_nop 4" : "+v"(w), "+v"(off), "+v"(owed));      // DPP operands: not within two cycles of a vector write
        step4<0, 4>(base, off, xA, owed, xB, acc);
        step4<4, 8>(base, off, xB, owed, xC, acc);
        step4<8, 12>(base, off, xC, owed, xD, acc);
        step4<12, 0>(base, off, xD, w, xA, acc);
        owed = w;
    };
    for (uint32_t t = 0; t < a.nch; ++t) {
        if (t) {
            first_entries(t);
            __syncthreads();                                           // every wave has read what it needs of the last chunk
        }
        copy_window(t);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");             // this thread's part of the window is in LDS
        __syncthreads();
        // (no way out of the loop's middle: the compiler joins it to the loop's end, and every wait is then for all loads)
        const int2 *__restrict__ ahead = entries + (size_t)(g0 + kAhead) * 16u;
        uint32_t left = g1 - g0;
        for (; left >= kAhead; left -= kAhead, ahead += kAhead * 16u) {
#pragma unroll
            for (uint32_t i = 0; i < kAhead; ++i) {
                group(held[i]);
                held[i] = ahead[i * 16u + l16];
            }
        }
        rest<0>(left, [&](uint32_t i) { group(held[i]); });
    }
    asm volatile("s_nop 4" : "+v"(owed));
    fma4<4>(owed, xB, acc);
    fma4<8>(owed, xC, acc);
    fma4<12>(owed, xD, acc);

    if (live) {
        const size_t at = (((size_t)co * g.H_out + th0 + ty) * g.W_out + tw0 + tx) * B + b;
        if (resid) acc += resid[at];
        Y[at] = conv_epilogue<ACT>(acc, relu);
    }
}

template <int ACT>
__global__ __launch_bounds__(1024)
void conv2d_column_kernel(const int2 *__restrict__ entries, const uint32_t *__restrict__ first_group, ColArgs a, so_conv_geom g,
                          const float *__restrict__ X, uint32_t B, const float *__restrict__ bias,
                          const float *__restrict__ resid, float *__restrict__ Y)
{
    column_convolution<ACT>(entries, first_group, a, g, X, B, bias, resid, Y, blockIdx.x, blockIdx.y, false);
}

// Two convolutions of one input: the first's workgroups, then the second's.  Both read their operands from the arguments at a place that
// depends on which it is.
struct ColPair {
    ColCall call[2];
    const float *X;
    uint32_t B, wgs0, tiles[2], mTiles[2];
};
__global__ __launch_bounds__(1024)
void conv2d_column_pair_kernel(ColPair)
{
    const ColPair &p = *(const ColPair *)__builtin_amdgcn_kernarg_segment_ptr();
    const uint32_t which = blockIdx.x >= p.wgs0 ? 1u : 0u, id = blockIdx.x - (which ? p.wgs0 : 0u);
    const ColCall &c = p.call[which];
    const uint32_t tiles = p.tiles[which], block = window_div(id, tiles, p.mTiles[which]);
    column_convolution<kActNoneOrRelu>(c.entries, c.first_group, c.a, c.g, p.X, p.B, c.bias, nullptr, c.Y, id - block * tiles, block, c.relu != 0u);
}

template <int ACT>
void launch_columns(so_ctx *ctx, const so_conv_plan *plan, const ColArgs &a, dim3 grid, size_t lds, const float *dX, uint32_t B,
                    const float *dBias, const float *dResid, float *dY)
{
    const so_conv_columns &c = *so_conv_columns_for(plan, B);
    conv2d_column_kernel<ACT><<<grid, a.waves * 64u, lds, ctx->stream>>>(c.d_entries, c.d_first, a, plan->g, dX, B, dBias, dResid, dY);
}

constexpr uint64_t kColLds = 150 * 1024;

struct ColShape { uint32_t G, waves; size_t lds; double us, rounds; };

// Channels per workgroup by estimated time: rounds of workgroups over the chip, each with a start-up of 2.5 us and its
// longest chain at 10 ns per entry on a SIMD of its own, 7.5 ns per wave that shares it.  A large window is copied by
// more waves than compute.  Measured at batch 1 on a ResNet-18-shaped stack: 56x56x64 8.9 us, 28x28x128 8.1, 14x14x256
// 9.8, 7x7x512 14.4; the windowed kernel with the batch carried as four: 12.3, 14.1, 17.5, 27.6.  Of two sizes that the estimate holds equal the smaller where
// the larger fills the chip more than once: its start-ups run beside others' chains.  Of 242 layers of 20x20 to 260x260 at batch 1 to 3 that changes 54, none to
// the worse by more than the runs differ, by up to 1.6: 3 -> 64 at 224x224, 7x7/2, batch 1 15.3 -> 10.6 us, 6 -> 128 at 194x194, 5x5, 64.5 -> 42.6.  (Where the larger is
// resident at once the smaller copies more windows: 64 -> 64 at 56x56 8.0 -> 9.5.)
//
// From 8 entries on windows of few pixels are the rule, and many workgroups of few channels on large images: 2.75 us; a chunk's start-up by its
// LDS, 0.44 us and 24 ns per KB, 9 more for every further workgroup on the compute unit; 0.5 us for each of those, 2.2 for every further filling of the
// chip; chains at 8.3 ns an entry, 5.9 per wave.  Fitted on 500 layers of up to 128x128 and 512 channels at batches of 8, 16 and 32: half are
// within 7 %.
ColShape column_shape(const so_ctx *ctx, const so_conv_plan *plan, const so_conv_columns &c, uint32_t G)
{
    const double cus = ctx->compute_units, chain = (double)plan->E->total_nnz / plan->g.Cout + 8.0, tiles = (double)c.tiles_x * c.tiles_y;
    ColShape s{G, 0, (size_t)(c.cc + 1) * c.PE * c.batch * 4, 0.0, 0.0};
    s.waves = s.lds >= 48 * 1024 ? 16u : std::max(G, 8u);
    const double wgs = tiles * so_ceil_div(plan->g.Cout, G);
    const double fit = std::max<double>(1.0, std::min<double>(160 * 1024 / s.lds, 32 / s.waves));
    const double resident = std::min(fit, std::ceil(wgs / cus));
    s.rounds = std::ceil(wgs / (cus * fit));
    if (c.batch <= 4) {
        s.us = 3.0 + s.rounds * (2.5 + c.nch + chain * std::max(0.010, 0.0075 * std::max(1.0, resident * G / 4.0)));
    } else {
        const double start = c.nch * (0.44 + 0.024 * s.lds / 1024.0 * (1.0 + 0.38 * (resident - 1.0))), waves = std::min(G, plan->g.Cout);
        s.us = 2.75 + s.rounds * (start + chain * std::max(0.0083, 0.0059 * std::max(1.0, resident * waves / 4.0))) +
               2.2 * std::max(0.0, wgs / (cus * fit) - 1.0) + 0.5 * (resident - 1.0);
    }
    return s;
}

ColShape column_shape(const so_ctx *ctx, const so_conv_plan *plan, const so_conv_columns &c)
{
    ColShape best{16, 16, 0, 1e30, 1.0};
    for (uint32_t G = 16; G >= 4; G /= 2)
        if (const ColShape s = column_shape(ctx, plan, c, G); s.us < best.us || (s.us == best.us && best.rounds > 1.0)) best = s;
    return best;
}

} // namespace

void so_conv_columns_free(so_conv_plan *plan)
{
    for (so_conv_columns &c : plan->col) {
        if (c.d_entries) (void)hipFree(c.d_entries);
        if (c.d_first) (void)hipFree(c.d_first);
        c = so_conv_columns();
    }
}

const so_conv_columns *so_conv_columns_for(const so_conv_plan *plan, uint32_t B)
{
    const int slot = so_conv_columns_slot(B);
    return slot >= 0 && plan->col[slot].batch == B ? &plan->col[slot] : nullptr;
}

// The tile and the window for batch B, without streams; false where the kernel does not apply.
static bool columns_geometry(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B, so_conv_columns &c)
{
    const so_conv_geom &g = plan->g;
    const so_ellpack *E = plan->E;
    if (so_conv_columns_slot(B) < 0 || E->r == 0 || E->total_nnz == 0 || !E->ascending || (size_t)ctx->max_lds_bytes < kColLds) return false;
    const uint32_t px = 64u / B, sth = window_step(g.kH, g.stride_h), stw = window_step(g.kW, g.stride_w);
    uint64_t best_tiles = ~0ull, best_win = ~0ull;
    for (uint32_t th = 1; th <= px && th <= g.H_out; ++th)
        for (uint32_t tw = 1; th * tw <= px && tw <= g.W_out; ++tw) {
            const uint64_t tiles = (uint64_t)so_ceil_div(g.H_out, th) * so_ceil_div(g.W_out, tw);
            const uint64_t win = (uint64_t)((th - 1) * sth + (g.kH - 1) * g.dil_h + 1) * ((tw - 1) * stw + (g.kW - 1) * g.dil_w + 1);
            if (tiles < best_tiles || (tiles == best_tiles && win < best_win)) { best_tiles = tiles; best_win = win; c.TH = th; c.TW = tw; }
        }
    if (c.TH == 0) return false;
    c.tiles_x = so_ceil_div(g.W_out, c.TW);
    c.tiles_y = so_ceil_div(g.H_out, c.TH);
    const uint32_t IH = (c.TH - 1) * sth + (g.kH - 1) * g.dil_h + 1, IW = (c.TW - 1) * stw + (g.kW - 1) * g.dil_w + 1;
    // A tile as wide as the image whose first and last window columns both lie outside it: the last column of a row and
    // the first of the next, zeros both, share their place (7 x 7 x 512: 147 KB instead of 166, one chunk instead of two).
    const bool share = c.tiles_x == 1 && IW > 1 && g.pad_w >= 1 && g.kW > 1 && (uint64_t)IW - 1 >= (uint64_t)g.W_in + g.pad_w;
    c.IP = share ? IW - 1 : IW;
    c.PE = (IH - 1) * c.IP + IW;
    const uint64_t plane = (uint64_t)c.PE * B;
    if (plane * 4 * 2 > kColLds) return false;
    c.cc = (uint32_t)std::min<uint64_t>(g.Cin, kColLds / (plane * 4) - 1);
    c.nch = so_ceil_div(g.Cin, c.cc);
    c.cc = so_ceil_div(g.Cin, c.nch);
    // window_div: operand * divisor below 2^32
    if ((uint64_t)c.tiles_x * c.tiles_x * c.tiles_y >= (1ull << 32) || plane * plane >= (1ull << 32) || plane * 1024 >= (1ull << 32)) return false;
    if ((uint64_t)c.tiles_x * c.tiles_y >= (1ull << 31) || ((uint64_t)c.cc + 1024) * g.H_in * g.W_in * B >= (1ull << 30)) return false;
    c.batch = B;
    return true;
}

// At more than four entries no streams for a plan whose windowed layout the kernel would not be taken before: looked at anew by every tuning,
// since the layout and the overrides may be others by then.
bool so_conv_columns_wanted(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B)
{
    so_conv_columns c;
    if (!columns_geometry(ctx, plan, B, c)) return false;
    return B <= 4 || ctx->tune.conv_columns == 1 || so_conv_columns_before_window(ctx, plan, B, column_shape(ctx, plan, c).us);
}

// Uploads the entry streams for batch B; leaves the plan without them where the kernel does not apply.
so_status so_conv_columns_build(so_ctx *ctx, so_conv_plan *plan, const std::vector<uint32_t> &idx, const std::vector<uint32_t> &nnz,
                                const std::vector<float> &Wd, uint32_t B)
{
    const so_conv_geom &g = plan->g;
    const so_ellpack *E = plan->E;
    so_conv_columns c;
    if (!columns_geometry(ctx, plan, B, c)) return SO_OK;
    const uint64_t plane = (uint64_t)c.PE * B;
    const uint32_t kHW = g.kH * g.kW;
    const size_t runs = (size_t)E->m * c.nch;
    std::vector<uint32_t> first(runs + 1);      // entries of every (channel, chunk), then groups, then where they begin
    for (uint32_t co = 0; co < E->m; ++co)
        for (uint32_t j = 0; j < nnz[co]; ++j) ++first[(size_t)co * c.nch + idx[(size_t)co * E->r + j] / kHW / c.cc];
    uint64_t total = 0;
    for (uint32_t &f : first) { f = (f + 15u) / 16u; total += f; c.pitch = std::max(c.pitch, f); }
    // at a pitch unless few long runs make that much larger
    if ((uint64_t)runs * c.pitch > 2 * total + 1024) c.pitch = 0;
    else total = (uint64_t)runs * c.pitch;
    if (total > 0xfffffff0ull) return SO_OK;
    uint32_t pad_bits;
    const float neg_zero = -0.0f;
    std::memcpy(&pad_bits, &neg_zero, 4);
    std::vector<int2> entries(((size_t)total + kAhead) * 16, make_int2((int)pad_bits, (int)(c.cc * plane * 4)));
    size_t next = 0;                            // group
    for (uint32_t co = 0; co < E->m; ++co) {
        uint32_t j = 0;
        for (uint32_t t = 0; t < c.nch; ++t) {
            const size_t run = (size_t)co * c.nch + t;
            if (c.pitch) next = run * c.pitch;
            int2 *e = entries.data() + next * 16;
            for (; j < nnz[co]; ++j) {
                const size_t slot = (size_t)co * E->r + j;
                const uint32_t k = idx[slot], cin = k / kHW, kh = (k / g.kW) % g.kH, kw = k % g.kW;
                if (cin >= (t + 1) * c.cc) break;
                uint32_t wb;
                std::memcpy(&wb, &Wd[slot], 4);
                *e++ = make_int2((int)wb, (int)(((uint64_t)(cin - t * c.cc) * plane + (uint64_t)(kh * g.dil_h * c.IP + kw * g.dil_w) * B) * 4));
            }
            if (!c.pitch) { const uint32_t groups = first[run]; first[run] = (uint32_t)next; next += groups; }
        }
    }
    if (!c.pitch) first.back() = (uint32_t)next;
    for (const void *k : {(const void *)conv2d_column_kernel<SO_ACT_NONE>, (const void *)conv2d_column_kernel<SO_ACT_RELU>,
                          (const void *)conv2d_column_kernel<SO_ACT_SIGMOID>, (const void *)conv2d_column_kernel<SO_ACT_TANH>, (const void *)conv2d_column_pair_kernel})
        SO_HIP(so_allow_big_lds(ctx, k));
    void *p = nullptr;
    so_status s = so_malloc(ctx, entries.size() * sizeof(int2), &p);
    if (s != SO_OK) return s;
    c.d_entries = (int2 *)p;
    if ((s = so_malloc(ctx, first.size() * 4, &p)) == SO_OK) {
        c.d_first = (uint32_t *)p;
        s = so_h2d(ctx, c.d_entries, entries.data(), entries.size() * sizeof(int2));
        if (s == SO_OK) s = so_h2d(ctx, c.d_first, first.data(), first.size() * 4);
    }
    if (s != SO_OK) {
        (void)hipFree(c.d_entries);
        if (c.d_first) (void)hipFree(c.d_first);
        return s;
    }
    plan->col[so_conv_columns_slot(B)] = c;
    return SO_OK;
}

// Whether the kernel is taken before the gather kernel: both walk a channel's entries for every output, this one after a
// copy of the window, which entries enough repay -- more of them where the gather kernel has two or four batch entries to
// fetch at once, or no taps that share cache lines to fetch them from.  us, gather kernel / this one, at batch 1 and 2:
//   one round of workgroups: 64 x 56 x 56 -> 64, 3x3, 116 entries a channel 21.2 / 8.5 and 22.7 / 13.3; 7 -> 8 at 31 x 30, 3x3/2, 31 entries
//   6.7 / 3.7 and 6.8 / 4.1; 5 -> 47 at 14 x 10, 3x3/2, 9 entries 4.1 / 3.4 and 4.1 / 3.5; 4 -> 314 at 34 x 38, 1x1/2, 4 entries
//   3.3 / 3.5 and 3.4 / 4.8; a large window for few entries: 587 -> 359 at 19 x 17, 1x1/2, 30 entries 6.8 / 8.8 and 5.5 / 13.4,
//   106 -> 41 at 123 x 150, 3x3/2, 48 entries 13.1 / 14.9 and 17.8 / 42;
//   more rounds, 3x3 to 7x7: 3 -> 16 at 512 x 512, 12 entries 37.5 / 29.0 and 40.6 / 55.0; 3 -> 32 at 1000 x 1000, 16 entries 215 / 210;
//   7 -> 220 at 450 x 450, /2, 32 entries 163 / 110 and 173 / 184; 17 -> 5 at 600 x 600, /2, 75 entries 28.1 / 13.7 and 26.9 / 21.2; 3 -> 64 at 224 x 224, 15 entries
//   28.7 / 22.7 and 31.6 / 40.5; 3 -> 48 at 160 x 160, 7x7/2, 45 entries, batch 2 13.1 / 8.1; 5 -> 173 at 219 x 219, 5x5, 44 entries, batch 2 166 / 120; with many channels in
//   the window 64 -> 64 at 300 x 300, 17 entries 64 / 123 and 99 / 229;
//   34 -> 116 at 160 x 207, 168 entries 224 / 91 and 327 / 228; 1x1: 33 -> 197 at 509 x 526, /2, 10 entries 97 / 695 and 131 / 1121; 63 -> 74
//   at 92 x 74, 63 entries 13.4 / 14.8 and 20 / 27; 214 -> 12 at 77 x 77, 214 entries 21.8 / 10.2 and 29.6 / 9.4.  At batch 4 (plans without
//   the windowed layout): 72 entries 133 / 170, 75 29.5 / 28.0, 118 54.5 / 46.6, 147 79 / 72.
bool so_conv_columns_pays(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B)
{
    const so_conv_columns &c = *so_conv_columns_for(plan, B);
    const double entries = (double)plan->E->total_nnz / plan->g.Cout, window = (double)c.cc * c.nch * c.PE * B;
    if (entries < 8.0 || window > 480.0 * entries) return false;
    const bool taps = plan->g.kH * plan->g.kW > 1;
    const double least = B == 4 ? 100.0 : B == 2 || !taps ? 64.0 : 20.0;
    if (entries >= least || column_shape(ctx, plan, c).rounds <= 1.0) return true;
    return taps && B < 4 && entries >= (B == 2 ? 40.0 : 14.0) && window <= 100.0 * entries;
}

double so_conv_columns_estimate(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B) { return column_shape(ctx, plan, *so_conv_columns_for(plan, B)).us; }

// The arguments of a launch; false: the kernel does not take it.
static bool columns_arguments(const so_conv_plan *plan, const so_conv_columns &c, const ColShape &shape, ColArgs &a, dim3 &grid)
{
    const so_conv_geom &g = plan->g;
    const uint32_t B = c.batch;
    a.TH = c.TH; a.TW = c.TW; a.tiles_x = c.tiles_x; a.PE = c.PE; a.IP = c.IP; a.PL = c.PE * B; a.cc = c.cc; a.nch = c.nch; a.pitch = c.pitch;
    a.sth = window_step(g.kH, g.stride_h); a.stw = window_step(g.kW, g.stride_w);
    a.sbh = window_subsample(g.kH, g.stride_h); a.sbw = window_subsample(g.kW, g.stride_w);
    a.mB = window_magic(B); a.mIP = window_magic(a.IP); a.mPL = window_magic(a.PL); a.mTW = window_magic(a.TW); a.mTilesX = window_magic(a.tiles_x);
    a.G = shape.G;
    a.waves = shape.waves;
    grid = dim3(c.tiles_x * c.tiles_y, so_ceil_div(g.Cout, a.G));
    return grid.y <= 65535u;
}

so_status so_conv_columns_launch(so_ctx *ctx, const so_conv_plan *plan, const float *dX, uint32_t B, const float *dBias,
                                 const float *dResid, float *dY, int act, bool *done)
{
    *done = false;
    if (!so_conv_columns_for(plan, B)) return SO_OK;
    const so_conv_columns &c = *so_conv_columns_for(plan, B);
    const ColShape shape = column_shape(ctx, plan, c);
    const size_t lds = shape.lds;
    ColArgs a;
    dim3 grid;
    if (!columns_arguments(plan, c, shape, a, grid)) return SO_OK;
    *done = true;
    switch (act) {
    case SO_ACT_RELU:    launch_columns<SO_ACT_RELU>(ctx, plan, a, grid, lds, dX, B, dBias, dResid, dY); break;
    case SO_ACT_SIGMOID: launch_columns<SO_ACT_SIGMOID>(ctx, plan, a, grid, lds, dX, B, dBias, dResid, dY); break;
    case SO_ACT_TANH:    launch_columns<SO_ACT_TANH>(ctx, plan, a, grid, lds, dX, B, dBias, dResid, dY); break;
    default:             launch_columns<SO_ACT_NONE>(ctx, plan, a, grid, lds, dX, B, dBias, dResid, dY); break;
    }
    return SO_OK;
}

// A launch of its own for a residual block's projection is mostly start-up.  Here its workgroups run beside the first convolution's where the sizes that are
// chosen for both let all be resident at once -- the longer of the two is the time -- and behind them otherwise, where each alone is one filling of the chip at
// the occupancy that the larger window leaves: then a launch's gap is saved.  Us, ResNet-18-shaped stacks, one after the other / together: 224x224 of width 64
// at batch 1 8.3 + 4.4 / 9.4, 10.6 + 5.1 / 14.1, 16.2 + 5.5 / 16.6, at 8 (into 7x7) 31.2 + 7.1 / 34.6; 96x96 of 64 at 8 12.3 + 5.1 / 12.8,
// 13.4 + 5.1 / 14.0, 17.6 + 5.9 / 22.7.
so_status so_conv_columns_launch_pair(so_ctx *ctx, const so_conv_call (&call)[2], const float *dX, uint32_t B, bool *done)
{
    *done = false;
    const so_conv_columns *const c[2] = {so_conv_columns_for(call[0].plan, B), so_conv_columns_for(call[1].plan, B)};
    if (!c[0] || !c[1]) return SO_OK;
    double best = column_shape(ctx, call[0].plan, *c[0]).us + column_shape(ctx, call[1].plan, *c[1]).us;
    ColPair p;
    uint32_t wgs = 0, waves = 0;
    size_t lds = 0;
    for (uint32_t G0 = 16; G0 >= 4; G0 /= 2)
        for (uint32_t G1 = 16; G1 >= 4; G1 /= 2) {
            const ColShape s[2] = {column_shape(ctx, call[0].plan, *c[0], G0), column_shape(ctx, call[1].plan, *c[1], G1)};
            ColArgs a[2];
            dim3 grid[2];
            if (!columns_arguments(call[0].plan, *c[0], s[0], a[0], grid[0]) || !columns_arguments(call[1].plan, *c[1], s[1], a[1], grid[1])) continue;
            const size_t most = std::max(s[0].lds, s[1].lds);
            const uint32_t w = std::max(s[0].waves, s[1].waves);
            const uint64_t one = (uint64_t)grid[0].x * grid[0].y, two = (uint64_t)grid[1].x * grid[1].y, all = one + two;
            const uint64_t resident = (uint64_t)ctx->compute_units * std::max<uint64_t>(1, std::min<uint64_t>(160 * 1024 / most, 32 / w));
            if (one > resident || two > resident) continue;
            const double us = all <= resident ? std::max(s[0].us, s[1].us) : s[0].us + s[1].us - 2.0;
            if (us >= best) continue;
            best = us; wgs = (uint32_t)all; waves = w; lds = most;
            p.wgs0 = grid[0].x * grid[0].y;
            for (int i = 0; i < 2; ++i) {
                a[i].waves = w;
                p.call[i].a = a[i];
                p.tiles[i] = grid[i].x; p.mTiles[i] = window_magic(grid[i].x);
            }
        }
    if (!wgs) return SO_OK;
    for (int i = 0; i < 2; ++i) {
        ColCall &o = p.call[i];
        o.entries = c[i]->d_entries; o.first_group = c[i]->d_first;
        o.bias = call[i].dBias; o.Y = call[i].dY;
        o.g = call[i].plan->g;
        o.relu = call[i].act == SO_ACT_RELU;
    }
    p.X = dX; p.B = B;
    conv2d_column_pair_kernel<<<wgs, waves * 64u, lds, ctx->stream>>>(p);
    *done = true;
    return SO_OK;
}
