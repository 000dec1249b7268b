// Internal definitions shared by the HIP translation units of libsparseops_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "parallel.h"
#include "sparseops_hip.h"

// Tuning overrides, read from the environment when the context is created (and again by
// so_tuning_reload), never per launch.  0 / -1 = the library's own choice.
struct so_tuning {
    int matmul_tiled = -1;   // SPARSEOPS_MATMUL_TILED: 1 forces the LDS-staged kernel, 0 forbids it
    int matmul_vec = 0;      // SPARSEOPS_MATMUL_VEC: 1 or 2 columns per lane at most
    int matmul_share = -1;   // SPARSEOPS_MATMUL_SHARE: 0 forbids the shared-gather kernel for few-row launches
    int matmul_columns = -1; // SPARSEOPS_MATMUL_COLUMNS: 0 forbids the kernel with X in LDS for few columns, 1 forces it where it applies
    int matmul_rbm = -1;     // SPARSEOPS_MATMUL_RBM: 0 forbids every kernel that is only for handles with the RBM layout, 1 forces the row-block-merged one
    int matmul_rbm_split = 0;   // SPARSEOPS_MATMUL_RBM_SPLIT: 1, 2 or 4 workgroups per tile for RBM layouts built from now on
    int matmul_quad = -1;    // SPARSEOPS_MATMUL_QUAD: 0 forbids the quad-union kernel on handles with the RBM layout, 1 forces it
    int matmul_quad_rows = -1;  // SPARSEOPS_MATMUL_QUAD_ROWS: log2 of the quads per workgroup (0..4)
    int matmul_quad_split = 0;  // SPARSEOPS_MATMUL_QUAD_SPLIT: workgroups per output tile
    int matmul_narrow = -1;  // SPARSEOPS_MATMUL_NARROW: 0 forbids the narrow kernel on handles with the RBM layout, 1 forces it where it applies
    int matmul_slabs = -1;   // SPARSEOPS_MATMUL_SLABS: 0 forbids the quad-union copy's kernel with X in LDS a part at a time, 4 and 8 force it where it applies, with slabs of 16 and 32 columns
    int matmul_planes = -1;  // SPARSEOPS_MATMUL_PLANES: 0 forbids the bf16-planes kernel on handles with the RBM layout, 1 forces it where the handle has the planes
    int matmul_planes_split = 0;   // SPARSEOPS_MATMUL_PLANES_SPLIT: workgroups per output tile
    int matvec_lanes = 0;    // SPARSEOPS_MATVEC_LANES: 8, 16, 32 or 64 lanes per row
    int matvec_idx16 = -1;   // SPARSEOPS_MATVEC_IDX16: 0 keeps so_matvec on the 32-bit columns of a handle that has both
    int conv_min_cg = 0;     // SPARSEOPS_CONV_MIN_CG: fewest channel groups per workgroup a small grid may shrink to (16: never shrink)
    int conv_window = -1;    // SPARSEOPS_CONV_WINDOW: 1 forces the LDS-windowed kernel, 0 forbids it
    int conv_cpw = 0;        // SPARSEOPS_CONV_CPW: most output channels per wave
    int conv_tilepx = 0;     // SPARSEOPS_CONV_TILEPX: most output pixels per tile
    int conv_columns = -1;   // SPARSEOPS_CONV_COLUMNS: 0 forbids the column kernel, 1 forces it on plans tuned for the batch
    int conv_vec = 0;        // SPARSEOPS_CONV_VEC: most batch entries per lane in the gather kernel
    int wait_spins = -1;     // SPARSEOPS_WAIT_SPINS: most polls of a bounded wait on LDS progress counters (0: every wait gives up at once; tests)
    int conv_rbm = -1;       // SPARSEOPS_CONV_RBM: 0 forbids the row-block-merged kernel on plans that carry its streams, 1 asks for it against any other override
};

// Device memory that the library may replace by itself (a workspace that grows, a layout that is rewritten): its kernels
// get the address as an argument, so a recorded graph replays with it.  Owned together by whoever uses it now and by
// every graph recorded with it, and freed with the last of them.
struct so_block {
    void *p = nullptr;
    size_t bytes = 0;
    so_block() = default;
    so_block(const so_block &) = delete;
    so_block &operator=(const so_block &) = delete;
    ~so_block() { if (p) (void)hipFree(p); }
};
using so_block_ref = std::shared_ptr<so_block>;

constexpr uint64_t kEncodeSpareFirst = 1ull << 30, kEncodeSpareMost = 1ull << 34;

struct so_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int compute_units = 0;
    int max_lds_bytes = 0;   // largest LDS allocation one workgroup may ask for
    bool capturing = false;
    void *static_scratch = nullptr;   // this device's address of the library's static scratch array (so_ellpack_encode_noalloc)
    // Bounded waits (csrc/lds_sync.h): a device word in which waves that gave up count themselves, its pinned
    // host copy, and whether a kernel that waits that way has been launched since the word was last looked at.
    uint32_t *d_wait_gave_up = nullptr;
    uint32_t *h_wait_gave_up = nullptr;
    bool waits_pending = false;
    uint32_t *h_encode_header = nullptr;   // pinned: {r, total nnz (low, high)} of the last encode that asked for them
    // After a one-read encode whose workgroups gave up waiting for one another: elements still to be encoded in two passes, and how many the next time
    uint64_t encode_spared = 0, encode_spare_next = kEncodeSpareFirst;
    // Staging of host arrays (so_stage_in, so_stage_out): pinned memory, the flag of the last way out in it, its bytes in use
    char *h_stage = nullptr;
    uint32_t *d_stage_done = nullptr;      // workgroups of a way out that have finished
    size_t stage_used = 0;
    uint32_t stage_turn = 0;
    uint32_t told_turn = 0;                // of the word behind the encoder's header in h_wait_gave_up's memory
    // Workspace of so_matmul's kernels that split a tile over workgroups: partial tiles, a zeroed counter per tile
    so_block_ref mm_part, mm_counters;
    std::vector<so_block_ref> recorded;          // what the launches of the recording under way use (so_keep_recorded)
    std::string name;
    so_tuning tune;
    const char *last_kernel = "";                // so_last_kernel
    std::vector<const void *> big_lds_kernels;   // kernels already allowed max_lds_bytes of dynamic LDS on this device
};

// Rows of one length class for the binned matvec: `group` lanes cooperate on a row.
constexpr uint32_t kStagePairsMost = 8192;       // floats of a result that goes to the staging memory as pairs {value, turn}

struct so_bin {
    uint32_t group = 0;      // 4, 16 or 64 lanes per row, 1024: a whole workgroup
    uint32_t count = 0;      // rows in this class
    uint32_t *d_rows = nullptr;   // count pairs (row, nonzeros of the row), longest rows first
};

// K-tiled copy of the matrix for the LDS-staged matmul.  Rows are grouped in
// quads (four rows share a wavefront, 16 lanes each); the dense operand is consumed
// in tiles of kTileRows rows.  For every (quad, tile) the nonzeros whose column
// falls in the tile are stored as "steps": step s holds one (weight, LDS byte
// offset of the X row inside the tile) pair per row of the quad, padded with
// (0, offset of a zero row) for rows that have fewer nonzeros in this tile.
// Steps are stored in chunks of 16: chunk[g][k] is the pair of row g for step k,
// so the 64 lanes of a wave fetch one chunk with a single coalesced 8-byte load.
struct so_tile_entry { float w; uint32_t off; };
struct so_tile_info { uint32_t chunk0; uint32_t steps; };   // steps is a multiple of 4
struct so_tiled {
    static constexpr uint32_t kTileRows = 256;   // X rows per LDS tile
    static constexpr uint32_t kWavesPerGroup = 16;   // quads (waves) per workgroup of the kernel
    static constexpr uint32_t kSlabCols = 64;    // dense columns per workgroup
    static constexpr uint32_t kTileBytes = kTileRows * kSlabCols * 4;
    static constexpr uint32_t kZeroRowOff = 2 * kTileBytes;      // after the two tile buffers
    static constexpr uint32_t kSyncOff = kZeroRowOff + kSlabCols * 4;    // the workgroup's progress counters (csrc/lds_sync.h)
    static constexpr uint32_t kLdsBytes = kSyncOff + 64;
    uint32_t nquads = 0, ntiles = 0;
    uint64_t total_steps = 0;
    so_tile_entry *d_entries = nullptr;   // [chunks + 3][64]
    so_tile_info *d_info = nullptr;       // [nquads][ntiles]
    uint32_t *d_rows = nullptr;           // [nquads*4] row id of each quad member (0xffffffff = none)
};

// Row-block-merged copy of the matrix for so_matmul (csrc/matmul_rbm.hip): per block of 128 rows and per
// stream (12 waves x ksplit workgroups) a run of 256-byte records, one per loop iteration, and at the same
// index of `w` the iteration's 64 weights.
struct so_rbmm {
    static constexpr uint32_t kBlockRows = 128;   // rows (accumulators) per tile
    static constexpr uint32_t kWaves = 12;        // waves per workgroup
    static constexpr uint32_t kMaxSplit = 4;      // most workgroups per tile
    uint32_t nb = 0, ksplit = 1;
    uint64_t nrec = 0;                            // records (= weight blocks), tails included
    uint64_t slots = 0, xloads = 0;               // multiply-adds a 64-column slab costs (padding included), X row segments it loads
    void *d_blob = nullptr;                       // one allocation for the arrays below
    uint32_t *d_hdr = nullptr;                    // per block: iterations per class (6 dwords + 2 spare), then per stream {first record, first class}
    uint32_t *d_rec = nullptr;
    float *d_w = nullptr;
    uint32_t *d_xrows = nullptr;                  // [nrec][4]: the X rows of every record; the records hold row * pitch
    so_block_ref recs;                            // owner of d_rec where set_pitch moved it; else empty, held by graphs recorded with d_rec all the same
    uint32_t pitch = 0;                           // row pitch of X (bytes) the records' offsets are written for; 0: none yet
};

// Quad-union copy of the matrix for so_matmul on the matrix cores (csrc/matmul_quad.hip): four consecutive rows
// share a list of columns, cut by tiles of 256 columns and stored in chunks of 16 steps.
struct so_quads {
    static constexpr uint32_t kTileRows = 256;    // X rows per LDS tile
    static constexpr uint32_t kMaxSplit = 64;     // most workgroups per output tile
    static constexpr uint32_t kSlack = 128;       // chunks behind the last one that requests ahead may reach
    uint32_t nquads = 0, ntiles = 0;
    uint64_t total_units = 0, total_chunks = 0;   // units of four steps and chunks over all (quad, tile) runs
    float *d_w = nullptr;                         // [chunks + slack][64]
    uint32_t *d_off = nullptr;                    // [chunks + slack][4] words: X row inside the tile, a byte per step
    uint2 *d_info = nullptr;                      // [nquads][ntiles] {first chunk, units}
    static constexpr uint32_t kMostRows = 10240;  // X rows that the narrow kernel's LDS holds
    uint16_t *d_rows = nullptr;                   // [chunks + slack][16]: the X row of every step, for the narrow kernel (null beyond kMostRows columns)
};

// The matrix, dense, as three bf16 planes for so_matmul on the bf16 matrix cores (csrc/matmul_planes.hip).
struct so_planes {
    static constexpr uint32_t kMaxSplit = 16;     // most workgroups per output tile
    uint32_t k16 = 0;                             // runs of 16 columns kept per row tile
    void *d_a = nullptr;                          // [row tile of 32][k16][plane][64 lanes][8] bf16
};

struct so_ellpack {
    uint32_t m = 0, n = 0, r = 0;
    uint64_t total_nnz = 0;
    uint32_t max_nnz = 0;
    bool ascending = true;       // every row's stored columns are strictly ascending (what the encoder produces)
    int layouts = 0;
    float *d_Wd = nullptr;       // [m*r] row-major
    uint32_t *d_idx = nullptr;   // [m*r]
    uint32_t *d_nnz = nullptr;   // [m]
    float *d_WdT = nullptr;      // [r*m] slot-major (SO_LAYOUT_SLOT)
    uint32_t *d_idxT = nullptr;
    uint16_t *d_idx16 = nullptr; // [m*r] the columns of d_idx in 16 bits (SO_LAYOUT_IDX16, n <= 65536)
    uint16_t *d_idxT16 = nullptr;// [r*m] the same for d_idxT (SO_LAYOUT_SLOT with SO_LAYOUT_IDX16)
    so_bin bins[4];              // SO_LAYOUT_BINS
    std::vector<uint32_t> bin_order;   // their rows, the class of the longest first (kept up to kStagePairsMost rows)
    so_tiled tiled;              // SO_LAYOUT_TILED
    so_rbmm rbmm;                // SO_LAYOUT_RBM
    so_quads quads;              // SO_LAYOUT_RBM, unless the matrix is too sparse for it (d_w is null)
    so_planes planes;            // SO_LAYOUT_RBM, where so_planes_pays says so (else d_a is null)
};

// Row-block-merged re-encoding of a matrix (include/rbm_conv.hpp:8-27 of the reference), flattened:
// block b holds rows [b*Ct_max, min(M, (b+1)*Ct_max)); its union columns are krel[block_union[b] ..
// block_union[b+1]) in ascending order; union column u owns the pairs colptr[u] .. colptr[u+1], each
// a (row inside the block, weight), rows ascending.  Kept on the host: convolution plans turn it
// into the record streams their kernel reads.
struct so_rbm {
    uint32_t M = 0, N = 0, Ct_max = 0, nblocks = 0;
    std::vector<uint32_t> block_union, krel, colptr;
    std::vector<uint16_t> pair_row;
    std::vector<float> pair_w;
};

struct so_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<so_block_ref> uses;              // kept alive for the replays
};

void so_set_error(const char *fmt, ...);

// csrc/matmul_tiled.hip: launches the LDS-staged kernel on E's TILED copy (the caller has checked that it applies).
so_status so_matmul_tiled_launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C,
                                 const float *dBias, float *dY, int act);

// csrc/matmul_columns.hip: at most 64 dense columns with X in LDS, in the row kernels' order.
bool so_matmul_columns_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
double so_matmul_columns_estimate(const so_ctx *ctx, const so_ellpack *E, uint32_t C);      // us
so_status so_matmul_columns_launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY, int act);

// csrc/matmul_rbm.hip: the row-block-merged layout and its kernel.
so_status so_rbmm_build(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz);
void so_rbmm_free(so_ellpack *E);
bool so_matmul_rbm_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_rbm_set_pitch(so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_rbm_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_rbm_launch(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C,
                               const float *dBias, float *dY, int act);

// A block of `bytes` on the context's device (at least one).
so_status so_block_make(so_ctx *ctx, size_t bytes, so_block_ref *out);
// To be called for every block that a launch uses: while a graph is being recorded, the graph keeps it.
so_status so_keep_recorded(so_ctx *ctx, const so_block_ref &block);

// Grows the context's matmul workspace (partial tiles, a zeroed counter per tile).  Never while a graph is being recorded.
so_status so_matmul_workspace(so_ctx *ctx, size_t part_bytes, size_t counter_bytes);

// csrc/matvec.hip: the row kernel of so_matvec on each of C columns, with an activation.
so_status so_matvec_columns(so_ctx *ctx, const so_ellpack *E, const float *dX, uint32_t C, const float *dBias, float *dY, int act);

// csrc/matmul_quad.hip: the quad-union layout and its kernel.
so_status so_quads_build(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz);
void so_quads_free(so_ellpack *E);
// How a launch is split: quads per workgroup (log2), workgroups per output tile and the K tiles of each, slabs of 64 columns, row blocks.
struct so_quad_plan { uint32_t qw_log2, ks, tiles_per, nslab, rbs; double us; };
constexpr double kQuadLeastUs = 4.4;                                                  // no plan takes less (estimated)
bool so_matmul_quad_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_quad_plan so_matmul_quad_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
bool so_matmul_quad_ready(const so_ctx *ctx, const so_quad_plan &p);                  // the workspace need not grow for this launch
so_status so_matmul_quad_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_quad_launch(so_ctx *ctx, const so_ellpack *E, const so_quad_plan &p, const float *dX, uint32_t C,
                                const float *dBias, float *dY, int act);

// csrc/matmul_narrow.hip: few dense columns, or few rows, on the quad-union copy.
struct so_narrow_plan { uint32_t qw_log2, groups, slabs; bool passes; double us; };   // log2 of the quads per workgroup, 16-byte groups of a slab's row of X, slabs, X in LDS a part at a time
bool so_matmul_narrow_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_narrow_plan so_matmul_narrow_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
bool so_matmul_slabs_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);          // with X in LDS a part at a time
so_narrow_plan so_matmul_slabs_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_narrow_launch(so_ctx *ctx, const so_ellpack *E, const so_narrow_plan &p, const float *dX, uint32_t C, const float *dBias, float *dY, int act);

// csrc/matmul_planes.hip: the bf16 planes and their kernel.
struct so_planes_plan { uint32_t ks, iters, iters_per, nslab, mbs; double us; };   // workgroups per tile, iterations in all and of each, slabs, row blocks
bool so_planes_pays(const so_ctx *ctx, const so_ellpack *E);                              // csrc/matmul.hip: by estimate, some launch of the handle would take the kernel
so_status so_planes_build(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *nnz);
void so_planes_free(so_ellpack *E);
bool so_matmul_planes_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_planes_plan so_matmul_planes_choose(const so_ctx *ctx, uint32_t m, uint32_t n, uint32_t C);
bool so_matmul_planes_ready(const so_ctx *ctx, const so_planes_plan &p);                  // the workspace need not grow for this launch
so_status so_matmul_planes_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C);
so_status so_matmul_planes_launch(so_ctx *ctx, const so_ellpack *E, const so_planes_plan &p, const float *dX, uint32_t C,
                                  const float *dBias, float *dY, int act);

// csrc/encode_once.hip: encode from one read of the matrix.  `told` holds 2 * kEncodeTold words of 64 bits that nothing else writes;
// *done: launched, and once the host has been told (so_tell_wait) or, where *at_end then says so, the stream has ended host_header has
// {r, total nnz (low, high), 1 where it has to be done again}.
constexpr uint32_t kEncodeTold = 1024;
so_status so_encode_once(so_ctx *ctx, const float *dDense, uint32_t m, uint32_t n, uint32_t r_cap, uint32_t *dNnz, float *dWd, uint32_t *dIdx,
                         void *told, uint32_t *host_header, bool *done, volatile uint32_t **at_end);

// A launch that tells the host itself when its results are there: stored past the L2, so that the end of the kernel is not needed for others to see them.
struct so_tell {
    const uint32_t *gave_up;      // the context's word of bounded waits, for flag[1]
    uint32_t *flag;               // pinned: the turn, that word, one for the launch's own use
    uint32_t turn;
};
so_tell so_tell_next(so_ctx *ctx);
// Waits for such a launch, the context's last so_tell_next's, and reports as so_stream_wait does.
so_status so_tell_wait(so_ctx *ctx, const char *who);

template <typename T>
__device__ __forceinline__ void so_store_through(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// By a whole wave whose stores before it, also to the host, are to be there first.
__device__ __forceinline__ void so_tell_now(const so_tell &tell)
{
    if ((threadIdx.x & 63u) == 0) __hip_atomic_store(tell.flag + 1, __hip_atomic_load(tell.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    if ((threadIdx.x & 63u) == 0) __hip_atomic_store(tell.flag, tell.turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Waits for the context's stream and then reports, as SO_ERR_HIP, bounded waits that gave up in kernels launched
// since the last look (their results are invalid).  Every entry point that waits for the stream ends with this.
so_status so_stream_wait(so_ctx *ctx, const char *who);

// A result of up to kStagePairsMost floats that a launch itself writes to the staging memory, as a pair {value, turn} for each of them, and the wait for
// all of them.  False: there is no room, or no staging memory; *told false: the stream ended without them.
bool so_stage_result(so_ctx *ctx, uint32_t floats, uint2 **rows, uint32_t *turn);
so_status so_stage_result_take(so_ctx *ctx, uint32_t floats, const uint32_t *order, float *dst, uint32_t turn, bool *told);   // float i goes to dst[order[i]]

// Kernels that ask for more than 48 KB of dynamic LDS must be told so once per device: this does
// it the first time `kernel` is seen on the context's device (hipSuccess when already done).
hipError_t so_allow_big_lds(so_ctx *ctx, const void *kernel);

#define SO_HIP(call)                                                              \
    do {                                                                          \
        hipError_t e_ = (call);                                                   \
        if (e_ != hipSuccess) {                                                   \
            so_set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),   \
                         __FILE__, __LINE__);                                     \
            return e_ == hipErrorOutOfMemory ? SO_ERR_OOM : SO_ERR_HIP;           \
        }                                                                         \
    } while (0)

#define SO_REQUIRE(cond, ...)                                                     \
    do {                                                                          \
        if (!(cond)) {                                                            \
            so_set_error(__VA_ARGS__);                                            \
            return SO_ERR_INVALID;                                                \
        }                                                                         \
    } while (0)

// Launch check that is valid both eagerly and while a graph is being recorded.
#define SO_LAUNCH_CHECK()                                                         \
    do {                                                                          \
        hipError_t e_ = hipGetLastError();                                        \
        if (e_ != hipSuccess) {                                                   \
            so_set_error("kernel launch failed: %s (%s:%d)", hipGetErrorString(e_), \
                         __FILE__, __LINE__);                                     \
            return SO_ERR_HIP;                                                    \
        }                                                                         \
    } while (0)

static inline uint32_t so_ceil_div(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Epilogue shared by the matmul and conv kernels.  expf/tanhf are the accurate
// OCML routines (no fast-math), matching 1.0f/(1.0f+expf(-v)) and tanhf(v).
template <int ACT>
__device__ __forceinline__ float so_epilogue(float v)
{
    static_assert(ACT >= SO_ACT_NONE && ACT <= SO_ACT_TANH, "an activation");
    if (ACT == SO_ACT_RELU) return v > 0.0f ? v : 0.0f;
    if (ACT == SO_ACT_SIGMOID) return 1.0f / (1.0f + expf(-v));
    if (ACT == SO_ACT_TANH) return tanhf(v);
    return v;
}
