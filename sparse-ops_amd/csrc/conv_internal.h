// Definitions shared by the convolution translation units (conv.hip, conv_rbm.hip).
#pragma once

#include "so_internal.h"
#include "lds_sync.h"

#include <algorithm>
#include <vector>

// What the LDS-windowed kernel needs on top of the plan; built only for geometries it suits.
// The input channels are cut into chunks of `cc`; for one chunk and one tile of TH x TW output
// pixels the input window is IH x IW pixels.  A stored nonzero becomes the entry {weight bits,
// pixel offset of its tap inside the chunk's window}.  Output channels are taken `cpw` at a
// time (the channels one wave accumulates); the entries of such a channel group are one
// contiguous stream in the order the wave consumes them: chunk by chunk, inside a chunk channel
// by channel, inside a channel in slot order (slots are ordered by input channel, so a chunk is
// a slot range).  Every (chunk, channel) run is padded to a multiple of four entries with
// {-0.0, offset of an all-zero plane kept behind the window}: fma(-0, +0, acc) leaves any
// accumulator as it is.
struct so_conv_window {
    uint32_t planes = 1, PW = 0;  // column planes of a window row (PW columns, the last ones fewer): column iw lies at iw % planes * PW + iw / planes
    uint32_t TH = 0, TW = 0, IH = 0, IW = 0, cc = 0, nch = 0, tiles_x = 0, tiles_y = 0;
    uint32_t groups = 0;          // ceil(Cout / cpw)
    int cpw = 0;                  // output channels per wave
    uint32_t px = 1;              // pixel groups per wave where the batch tile is 16: 1 or 2
    uint32_t lpp = 0;             // lanes per pixel (batch tile / 4) the chunk size was chosen for: 4, 2 or 1
    int2 *d_stream = nullptr;     // all groups' streams, followed by one padding quad
    uint32_t *d_gbase = nullptr;  // [groups]: first quad (4 entries) of the group's stream
    uint32_t *d_quads = nullptr;  // [groups * nch * cpw]: quads of (group, chunk, channel in group)
};

// Record streams of the row-block-merged kernel (conv_rbm.hip) for the plan's current window layout.
struct so_conv_rbm {
    const so_rbm *src = nullptr;     // the attached format; must outlive the plan
    void *d_sets = nullptr;          // 64-byte sets of two records, all blocks, chunk after chunk
    uint32_t *d_gbase = nullptr;     // [blocks]: first set of the block's stream
    uint32_t *d_counts = nullptr;    // [blocks * chunks]: sets the loop walks for (block, chunk); 0: none
    uint64_t total_sets = 0, real_pairs = 0, slots = 0;
};

// Entry streams of the column kernel for small batches and small images (conv_columns.hip): batches of 1 to 4, 8, 16 and 32.
constexpr uint32_t kColSlots = 7;
inline int so_conv_columns_slot(uint32_t B) { return B >= 1 && B <= 4 ? (int)B - 1 : B == 8 ? 4 : B == 16 ? 5 : B == 32 ? 6 : -1; }
struct so_conv_columns {
    uint32_t batch = 0;              // the batch the tile and the offsets are for; 0: not built, or the kernel does not apply
    uint32_t TH = 0, TW = 0, tiles_x = 0, tiles_y = 0, IP = 0, PE = 0, cc = 0, nch = 0;
    uint32_t pitch = 0;              // groups from one (channel, chunk) to the next; 0: one right behind the other
    int2 *d_entries = nullptr;       // groups of 16 {weight bits, LDS byte offset}, channel by channel, chunk by chunk
    uint32_t *d_first = nullptr;     // [Cout * nch + 1]: groups of (channel, chunk) where there is a pitch, else its first group
};

struct so_conv_plan {
    uint32_t tuned_batch = 32;   // batch the windowed layout was sized for
    uint32_t tried_lpp = 0;      // lanes per pixel of the last attempt to build the windowed layout
    so_conv_geom g;
    const so_ellpack *E = nullptr;
    int2 *d_taps = nullptr;  // per slot: x = (cin*H + dh)*W + dw (elements of B floats), y = dh<<16 | (dw & 0xffff)
    so_conv_window win;      // win.cc == 0: not built
    so_conv_rbm rbm;         // rbm.d_sets == nullptr: no streams
    so_conv_columns col[kColSlots];      // streams by so_conv_columns_slot, made by the first tuning for the batch that wants them and kept: graphs may replay with them
    bool col_tried[kColSlots] = {};      // they have been made, or could not be
};

// Memory that nothing writes while a kernel runs, read by scalar loads also where the compiler does not see that by itself: behind inline assembly,
// through pointers that are not themselves the kernel's arguments.
template <class T> using so_constant = const __attribute__((address_space(4))) T *;

// One of the two convolutions of a so_conv2d_pair launch: what so_conv2d is given.
struct so_conv_call {
    const so_conv_plan *plan;
    const float *dBias;
    float *dY;
    int act;
};
// The pair kernels choose between the two activations that follow most convolutions when they run.
constexpr int kActNoneOrRelu = -1;
template <int ACT>
__device__ __forceinline__ float conv_epilogue(float v, bool relu)
{
    if constexpr (ACT == kActNoneOrRelu) return relu ? so_epilogue<SO_ACT_RELU>(v) : v;
    else return so_epilogue<ACT>(v);
}

// conv_columns.hip
void so_conv_columns_free(so_conv_plan *plan);
bool so_conv_columns_wanted(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B);          // streams for the batch pay
so_status so_conv_columns_build(so_ctx *ctx, so_conv_plan *plan, const std::vector<uint32_t> &idx, const std::vector<uint32_t> &nnz,
                                const std::vector<float> &Wd, uint32_t B);
const so_conv_columns *so_conv_columns_for(const so_conv_plan *plan, uint32_t B);  // null: the plan has no streams for the batch
bool so_conv_columns_pays(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B);            // against the gather kernel
double so_conv_columns_estimate(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B);      // us
bool so_conv_columns_before_window(const so_ctx *ctx, const so_conv_plan *plan, uint32_t B, double columns_us);   // conv.hip
so_status so_conv_columns_launch(so_ctx *ctx, const so_conv_plan *plan, const float *dX, uint32_t B, const float *dBias,
                                 const float *dResid, float *dY, int act, bool *done);
// Both of one input in one launch, where one is taken.
so_status so_conv_columns_launch_pair(so_ctx *ctx, const so_conv_call (&call)[2], const float *dX, uint32_t B, bool *done);

// conv_rbm.hip
void so_conv_rbm_release(so_conv_plan *plan);
so_status so_conv_rbm_rebuild(so_ctx *ctx, so_conv_plan *plan);
so_status so_conv_rbm_launch(so_ctx *ctx, const so_conv_plan *plan, const float *dX, uint32_t B, const float *dBias,
                             const float *dResid, float *dY, int act, bool *done);


constexpr int kWinThreads = 1024;
constexpr int kWinMaxPerThread = 6;   // float4 window elements a thread copies per chunk
constexpr uint32_t kWinLPP = 4;       // lanes per pixel of the preferred batch tile ...
constexpr uint32_t kWinBT = 4 * kWinLPP;   // ... of 16; batches that are only multiples of 8 or 4 use tiles of 8 or 4

// Lanes per pixel for batch B: the largest batch tile (16, 8, 4) that divides B; 0 if none does.
inline uint32_t window_lpp(uint32_t B) { return B % 16 == 0 ? 4u : B % 8 == 0 ? 2u : B % 4 == 0 ? 1u : 0u; }

struct WinArgs {
    uint32_t TH, TW, IH, IW, cc, nch, tiles_x, pg, cg, groups;
    uint32_t wgs, per_xcd;           // workgroups in all and per XCD (0: ids as launched)
    uint32_t yz, gz, mYZ = 0, oneYZ = 0, mZ = 0, oneZ = 0;   // (channel block, batch tile) pairs and batch tiles: window_magic, and all ones where that is one
    uint32_t win_f4;    // float4 elements of one chunk's window
    uint32_t buf_f4;    // window plus the zero plane: stride between the two buffers
    uint32_t nbuf;      // 2: double-buffered windows; 1: a single chunk, nothing to overlap
    uint32_t sth, stw;  // window pixels between neighbouring output pixels (stw: in a column plane)
    uint32_t planes, PW, mPW;   // so_conv_window::planes, the columns of one
    uint32_t sbh, sbw;  // input pixels between neighbouring window pixels
    uint32_t order[16]; // slot -> output pixel of the tile (ty * TW + tx), one byte per slot; see window_pixel_order
    uint32_t mIW, mIH, mTW, mTilesX, mPg;   // window_magic of IW, IH, TW, tiles_x and pg: the kernels' index arithmetic divides by them
    so_lds::wait_status ws;   // bounded waits on the progress counters
};

// x / d for the small operands of the window index arithmetic (x * d < 2^32: window elements and
// pixels count a few thousand, the divisors are window or tile extents) as one multiply-high by
// M = ceil(2^32 / d) instead of the ~25 instructions of a general 32-bit division: exact, because
// M * d - 2^32 < d makes the error of x * M / 2^32 smaller than 1 / d.  d == 1 has no 32-bit M.
inline uint32_t window_magic(uint32_t d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; }
__device__ __forceinline__ uint32_t window_div(uint32_t x, uint32_t d, uint32_t M) { return d == 1u ? x : __umulhi(x, M); }

// Along an axis on which the kernel has a single tap, a strided convolution reads only every
// stride-th input pixel: the window then holds just those (one window pixel per output pixel)
// instead of all the pixels in between.
inline uint32_t window_step(uint32_t k, uint32_t stride) { return k == 1 ? 1u : stride; }
inline uint32_t window_subsample(uint32_t k, uint32_t stride) { return k == 1 ? stride : 1u; }

// Workgroup ids go round the 8 XCDs; an XCD takes a contiguous share of the (tile, channel block, batch tile) triples, so that its L2
// holds an eighth of the input, whose halos neighbouring tiles share, and both halves of the 128-byte lines that two batch
// tiles of 16 read and write.  ResNet-18-shaped stack at batch 32, ids as (x, y, z) / so, us: 56x56x64 layers 45.8-51.1 / 43.7-47.0 (the
// write of 25.7 MB at the end of a layer 7 / 4), the stem 84.4 / 80.7, the stack 988 / 967.
//
// A launch has fewer than 2^32 work items along a dimension, so fewer than 2^22 workgroups of 1024: a grid whose product does not stay below
// that, or whose ids window_magic cannot divide, keeps them in (x, y, z), each of which then has to.
struct WinPlace { uint32_t tile, y, z; };
constexpr uint64_t kWinMaxGrid = (1ull << 32) / kWinThreads;
// Sets the shares for `grid`; the grid to launch is window_grid(a, grid).  False: no launch can have it.
inline bool window_shares(WinArgs &a, dim3 grid)
{
    if (grid.x >= kWinMaxGrid || grid.y > 65535u || grid.z > 65535u) return false;
    const uint64_t wgs = (uint64_t)grid.x * grid.y * grid.z, yz = (uint64_t)grid.y * grid.z;
    a.yz = (uint32_t)yz; a.gz = grid.z;
    a.wgs = a.per_xcd = 0;
    if ((wgs + 7) / 8 * 8 >= kWinMaxGrid || wgs * yz >= (1ull << 32) || yz * a.gz >= (1ull << 32)) return true;
    a.wgs = (uint32_t)wgs;
    a.per_xcd = (uint32_t)((wgs + 7) / 8);
    a.mYZ = window_magic((uint32_t)yz); a.oneYZ = yz == 1 ? ~0u : 0u;
    a.mZ = window_magic(a.gz); a.oneZ = a.gz == 1u ? ~0u : 0u;
    return true;
}
inline dim3 window_grid(const WinArgs &a, dim3 grid) { return a.per_xcd != 0u ? dim3(8u * a.per_xcd) : grid; }
__device__ __forceinline__ bool window_workgroup(const WinArgs &a, uint32_t wg, WinPlace &p)
{
    if (__builtin_expect(a.per_xcd == 0u, 0)) {
        p.tile = blockIdx.x; p.y = blockIdx.y; p.z = blockIdx.z;
        return true;
    }
    const uint32_t id = (wg & 7u) * a.per_xcd + (wg >> 3);
    p.tile = __umulhi(id, a.mYZ) + (id & a.oneYZ);
    const uint32_t rest = id - p.tile * a.yz;
    p.y = __umulhi(rest, a.mZ) + (rest & a.oneZ);
    p.z = rest - p.y * a.gz;
    return id < a.wgs;
}

// With an even stride along a row the lanes' reads of one tap would all fall on even (fourth, ...) window columns, half of the LDS's banks
// or less: the window's columns then lie in planes, those of one remainder by the stride side by side, so that neighbouring output
// pixels read neighbouring places.  ResNet-18-shaped layers at batch 32, one row / planes, us: stem 7x7/2 90 / 66 (80.5 on the
// row-block-merged kernel), 3x3/2 to 28x28x128 40.2 / 34.4, to 14x14x256 39.4 / 34.4, to 7x7x512 53 / 48.8; at batch 8 the stem 26.7 (merged) / 24.7.
//
// The input column of place `at` of a window row, from the window's first column on.
__device__ __forceinline__ uint32_t window_column(const WinArgs &a, uint32_t at)
{
    const uint32_t plane = __umulhi(at, a.mPW);                      // mPW is 0 for a single plane
    return __umul24(at - __umul24(plane, a.PW), a.planes) + plane;
}
// The same for a tap: where column kw of a tap lies, from an output pixel's corner on.
inline uint32_t window_tap_place(const so_conv_window &w, uint32_t kw) { return kw % w.planes * w.PW + kw / w.planes; }
inline void window_columns(WinArgs &a, const so_conv_window &w, const so_conv_geom &g)
{
    a.planes = w.planes; a.PW = w.PW; a.mPW = w.planes > 1 ? window_magic(a.PW) : 0u;
    a.stw = window_step(g.kW, g.stride_w) / w.planes;
}

// Which output pixel of the tile each pixel slot of the workgroup computes (slot = lanes / lanes per
// pixel, wave after wave).  LDS serves a 16-byte read 16 lanes at a time: 16 / lpp pixels, each a run
// of 16 * lpp bytes at (window pixel index) * 16 * lpp, i.e. on the bank group (window pixel index)
// mod (16 / lpp).  Pixels taken in row-major order collide on a bank group whenever the tile's rows
// are not a multiple of 16 / lpp pixels wide (tiles 7 pixels wide: every second read takes two
// turns).  Which slot computes which pixel is free, so the slots are dealt out such that the
// pixels of each group of 16 / lpp slots fall on different bank groups wherever the tile's shape
// allows it.  At most 64 pixels per tile; the table covers all 64 slots.
inline void window_pixel_order(WinArgs &a, uint32_t lpp)
{
    const uint32_t m = 16u / lpp, npx = a.TH * a.TW;
    std::vector<std::vector<uint8_t>> bucket(m);
    for (uint32_t p = 0; p < npx && p < 64u; ++p)
        bucket[((p / a.TW) * a.sth * a.IW + (p % a.TW) * a.stw) % m].push_back((uint8_t)p);
    for (auto &b : bucket) std::reverse(b.begin(), b.end());       // pop_back hands out the lowest pixel first
    uint8_t slots[64] = {0};
    uint32_t filled = 0;
    while (filled < npx && filled < 64u) {
        // one group: a pixel from each bank group, fullest first; then, if some are exhausted, more from the fullest
        std::vector<uint32_t> by_size(m);
        for (uint32_t r = 0; r < m; ++r) by_size[r] = r;
        std::stable_sort(by_size.begin(), by_size.end(), [&](uint32_t x, uint32_t y) { return bucket[x].size() > bucket[y].size(); });
        uint32_t taken = 0;
        for (uint32_t pass = 0; taken < m && filled < npx && filled < 64u; ++pass) {
            bool any = false;
            for (uint32_t k = 0; k < m && taken < m && filled < npx && filled < 64u; ++k) {
                std::vector<uint8_t> &b = bucket[by_size[k]];
                if (b.empty()) continue;
                slots[filled++] = b.back();
                b.pop_back();
                ++taken;
                any = true;
            }
            if (!any) break;
        }
    }
    // Slots beyond the tile compute nothing but still read: they repeat an address of their own group
    // of m slots (a read that several lanes share costs the banks one turn), or the previous group's.
    for (uint32_t i = filled; i < 64u; ++i) slots[i] = (i % m != 0) ? slots[i - i % m] : (i >= m ? slots[i - m] : 0);
    for (uint32_t i = 0; i < 16; ++i)
        a.order[i] = (uint32_t)slots[4 * i] | ((uint32_t)slots[4 * i + 1] << 8) | ((uint32_t)slots[4 * i + 2] << 16) | ((uint32_t)slots[4 * i + 3] << 24);
}

// The kernels' side: the output pixel of slot `pl` (< 64).
__device__ __forceinline__ uint32_t window_slot_pixel(const WinArgs &a, uint32_t pl)
{
    uint32_t word = 0;
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) word = (pl >> 2) == i ? a.order[i] : word;
    return (word >> ((pl & 3u) * 8u)) & 0xffu;
}
