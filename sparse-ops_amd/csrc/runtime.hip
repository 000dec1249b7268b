// Context, memory, timing, launch graphs and the device-resident ELLPACK layouts.
#include "so_internal.h"
#include "lane_moves.h"

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstring>
#include <exception>
#include <new>

static thread_local std::string g_last_error;

// Scratch memory of so_ellpack_encode_noalloc: the counting pass's header and per-workgroup partial
// results (layout further down, at the encoder), then the words of so_encode_once.  Every GPU the library runs on holds its own copy
// at its own address; host code never uses this name as a pointer, only the address that so_init
// looks up for the context's device.
constexpr size_t kEncodeToldOffset = 256 + 65536 * 8, kStaticScratchBytes = kEncodeToldOffset + kEncodeTold * 16;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

void so_set_error(const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

extern "C" const char *so_last_error(void) { return g_last_error.c_str(); }

extern "C" so_status so_device_count(int *n)
{
    SO_REQUIRE(n != nullptr, "so_device_count: n is null");
    *n = 0;
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess || c <= 0) {
        (void)hipGetLastError();
        so_set_error("no HIP device available (%s)", e == hipSuccess ? "count is 0" : hipGetErrorString(e));
        return SO_ERR_NO_DEVICE;
    }
    *n = c;
    return SO_OK;
}

hipError_t so_allow_big_lds(so_ctx *ctx, const void *kernel)
{
    for (const void *k : ctx->big_lds_kernels)
        if (k == kernel) return hipSuccess;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, ctx->max_lds_bytes);
    if (e == hipSuccess) ctx->big_lds_kernels.push_back(kernel);
    else (void)hipGetLastError();
    return e;
}

static int env_int(const char *name, int unset)
{
    const char *e = getenv(name);
    return (e && e[0]) ? atoi(e) : unset;
}

static void read_tuning(so_tuning &t)
{
    t = so_tuning();
    t.matmul_tiled = env_int("SPARSEOPS_MATMUL_TILED", -1);
    t.matmul_vec = env_int("SPARSEOPS_MATMUL_VEC", 0);
    t.matmul_share = env_int("SPARSEOPS_MATMUL_SHARE", -1);
    t.matmul_columns = env_int("SPARSEOPS_MATMUL_COLUMNS", -1);
    t.matmul_rbm = env_int("SPARSEOPS_MATMUL_RBM", -1);
    t.matmul_rbm_split = env_int("SPARSEOPS_MATMUL_RBM_SPLIT", 0);
    t.matmul_quad = env_int("SPARSEOPS_MATMUL_QUAD", -1);
    t.matmul_quad_rows = env_int("SPARSEOPS_MATMUL_QUAD_ROWS", -1);
    t.matmul_quad_split = env_int("SPARSEOPS_MATMUL_QUAD_SPLIT", 0);
    t.matmul_narrow = env_int("SPARSEOPS_MATMUL_NARROW", -1);
    t.matmul_slabs = env_int("SPARSEOPS_MATMUL_SLABS", -1);
    t.matmul_planes = env_int("SPARSEOPS_MATMUL_PLANES", -1);
    t.matmul_planes_split = env_int("SPARSEOPS_MATMUL_PLANES_SPLIT", 0);
    const int lanes = env_int("SPARSEOPS_MATVEC_LANES", 0);
    t.matvec_lanes = (lanes == 8 || lanes == 16 || lanes == 32 || lanes == 64) ? lanes : 0;
    t.matvec_idx16 = env_int("SPARSEOPS_MATVEC_IDX16", -1);
    t.conv_min_cg = env_int("SPARSEOPS_CONV_MIN_CG", 0);
    t.conv_window = env_int("SPARSEOPS_CONV_WINDOW", -1);
    t.conv_cpw = env_int("SPARSEOPS_CONV_CPW", 0);
    t.conv_tilepx = env_int("SPARSEOPS_CONV_TILEPX", 0);
    t.conv_vec = env_int("SPARSEOPS_CONV_VEC", 0);
    t.conv_columns = env_int("SPARSEOPS_CONV_COLUMNS", -1);
    t.conv_rbm = env_int("SPARSEOPS_CONV_RBM", -1);
    t.wait_spins = env_int("SPARSEOPS_WAIT_SPINS", -1);
}

extern "C" so_status so_tuning_reload(so_ctx *ctx)
{
    SO_REQUIRE(ctx != nullptr, "so_tuning_reload: ctx is null");
    read_tuning(ctx->tune);
    ctx->encode_spared = 0;                    // the bound of the waits may be another
    ctx->encode_spare_next = kEncodeSpareFirst;
    return SO_OK;
}

extern "C" so_status so_init(int device, so_ctx **out)
{
    SO_REQUIRE(out != nullptr, "so_init: out is null");
    *out = nullptr;
    int c = 0;
    so_status s = so_device_count(&c);
    if (s != SO_OK) return s;
    SO_REQUIRE(device >= 0 && device < c, "so_init: device %d out of range (have %d)", device, c);
    SO_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    SO_HIP(hipGetDeviceProperties(&prop, device));
    so_ctx *ctx = new (std::nothrow) so_ctx();
    if (!ctx) { so_set_error("so_init: host allocation failed"); return SO_ERR_OOM; }
    ctx->device = device;
    ctx->compute_units = prop.multiProcessorCount;
    ctx->max_lds_bytes = (int)prop.sharedMemPerBlock;
    ctx->name = prop.gcnArchName;
    read_tuning(ctx->tune);
    hipError_t e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev0);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev1);
    if (e != hipSuccess) {
        so_set_error("so_init: stream/event creation failed: %s", hipGetErrorString(e));
        so_destroy(ctx);
        return SO_ERR_HIP;
    }
    // this device's copy of the static scratch array (the device is current)
    e = hipGetSymbolAddress(&ctx->static_scratch, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ctx->static_scratch == nullptr) {
        so_set_error("so_init: hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        so_destroy(ctx);
        return SO_ERR_HIP;
    }
    // the word in which waves that give up a bounded wait count themselves, and its pinned host copy
    e = hipMalloc((void **)&ctx->d_wait_gave_up, 64);
    if (e == hipSuccess) e = hipMemset(ctx->d_wait_gave_up, 0, 64);
    if (e == hipSuccess) e = hipHostMalloc((void **)&ctx->h_wait_gave_up, 64, hipHostMallocCoherent);
    if (e != hipSuccess) {
        so_set_error("so_init: allocating the wait status word failed: %s", hipGetErrorString(e));
        so_destroy(ctx);
        return e == hipErrorOutOfMemory ? SO_ERR_OOM : SO_ERR_HIP;
    }
    std::memset(ctx->h_wait_gave_up, 0, 64);
    ctx->h_encode_header = ctx->h_wait_gave_up + 8;      // the same 64 bytes
    *out = ctx;
    return SO_OK;
}

// Waits for the stream; when a kernel with bounded waits has run since the last look, its status word
// comes back with the same wait (one 4-byte copy queued behind the work) and is cleared if it was set.
so_status so_stream_wait(so_ctx *ctx, const char *who)
{
    const bool look = ctx->waits_pending;
    if (look) SO_HIP(hipMemcpyAsync(ctx->h_wait_gave_up, ctx->d_wait_gave_up, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    SO_HIP(hipStreamSynchronize(ctx->stream));
    ctx->stage_used = 0;                       // nothing reads the staging memory any more
    if (!look) return SO_OK;
    ctx->waits_pending = false;
    const uint32_t gave_up = *ctx->h_wait_gave_up;
    if (gave_up == 0) return SO_OK;
    *ctx->h_wait_gave_up = 0;
    SO_HIP(hipMemsetAsync(ctx->d_wait_gave_up, 0, sizeof(uint32_t), ctx->stream));
    SO_HIP(hipStreamSynchronize(ctx->stream));
    so_set_error("%s: %u waits on LDS progress counters gave up in earlier launches; the results of those launches are invalid", who, gave_up);
    return SO_ERR_HIP;
}

extern "C" so_status so_destroy(so_ctx *ctx)
{
    if (!ctx) return SO_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) { (void)hipStreamSynchronize(ctx->stream); (void)hipStreamDestroy(ctx->stream); }
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    if (ctx->d_wait_gave_up) (void)hipFree(ctx->d_wait_gave_up);
    if (ctx->h_wait_gave_up) (void)hipHostFree(ctx->h_wait_gave_up);
    if (ctx->h_stage) (void)hipHostFree(ctx->h_stage);
    if (ctx->d_stage_done) (void)hipFree(ctx->d_stage_done);
    delete ctx;
    return SO_OK;
}

so_status so_block_make(so_ctx *ctx, size_t bytes, so_block_ref *out)
{
    try {
        so_block_ref b = std::make_shared<so_block>();
        SO_HIP(hipSetDevice(ctx->device));
        SO_HIP(hipMalloc(&b->p, std::max<size_t>(bytes, 4)));
        b->bytes = bytes;
        *out = std::move(b);
    } catch (const std::bad_alloc &) {
        so_set_error("host allocation failed");
        return SO_ERR_OOM;
    }
    return SO_OK;
}

so_status so_keep_recorded(so_ctx *ctx, const so_block_ref &block)
{
    if (!ctx->capturing || !block) return SO_OK;
    if (std::find(ctx->recorded.begin(), ctx->recorded.end(), block) != ctx->recorded.end()) return SO_OK;
    try {
        ctx->recorded.push_back(block);
    } catch (const std::bad_alloc &) {
        so_set_error("host allocation failed");
        return SO_ERR_OOM;
    }
    return SO_OK;
}

extern "C" const char *so_last_kernel(const so_ctx *ctx) { return ctx ? ctx->last_kernel : ""; }

extern "C" so_status so_device_info(so_ctx *ctx, char *name, size_t name_len, int *compute_units)
{
    SO_REQUIRE(ctx != nullptr, "so_device_info: ctx is null");
    if (name && name_len) {
        std::strncpy(name, ctx->name.c_str(), name_len - 1);
        name[name_len - 1] = '\0';
    }
    if (compute_units) *compute_units = ctx->compute_units;
    return SO_OK;
}

extern "C" so_status so_malloc(so_ctx *ctx, size_t bytes, void **dptr)
{
    SO_REQUIRE(ctx && dptr, "so_malloc: null argument");
    SO_REQUIRE(!ctx->capturing, "so_malloc: not allowed while a graph is being recorded");
    *dptr = nullptr;
    if (bytes == 0) bytes = 4;  // a valid, distinct pointer even for empty tensors
    SO_HIP(hipSetDevice(ctx->device));
    SO_HIP(hipMalloc(dptr, bytes));
    return SO_OK;
}

extern "C" so_status so_free(so_ctx *ctx, void *dptr)
{
    SO_REQUIRE(ctx != nullptr, "so_free: ctx is null");
    if (!dptr) return SO_OK;
    SO_REQUIRE(!ctx->capturing, "so_free: not allowed while a graph is being recorded");
    SO_HIP(hipStreamSynchronize(ctx->stream));
    SO_HIP(hipFree(dptr));
    return SO_OK;
}

extern "C" so_status so_h2d(so_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    SO_REQUIRE(ctx != nullptr, "so_h2d: ctx is null");
    if (bytes == 0) return SO_OK;
    SO_REQUIRE(dst && src, "so_h2d: null pointer");
    SO_REQUIRE(!ctx->capturing, "so_h2d: not allowed while a graph is being recorded");
    SO_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    return so_stream_wait(ctx, "so_h2d");
}

extern "C" so_status so_d2h(so_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    SO_REQUIRE(ctx != nullptr, "so_d2h: ctx is null");
    if (bytes == 0) return SO_OK;
    SO_REQUIRE(dst && src, "so_d2h: null pointer");
    SO_REQUIRE(!ctx->capturing, "so_d2h: not allowed while a graph is being recorded");
    SO_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    return so_stream_wait(ctx, "so_d2h");
}

// ---- staged copies: host arrays of calls that take and return host memory
//
// hipMemcpyAsync from and to pageable memory takes 15 us in and 21 us out for 4 KB, each with a wait of its own, and
// 34 and 42 us for 800 KB.  Here the host copies to pinned memory (4 KB 0.2 us, 800 KB 9 us) in pieces, and a kernel per
// piece reads that over the link while the next piece is copied; the way out is a kernel that writes pinned memory and
// then a word that the host polls.  Host to host, before and now: the MLP 784-4096-4096-4096-10 at batch 256 150 and 141 us, one image through the
// ResNet-18-shaped stack 312 and 284.
//
// Bound by latencies in a row: per kernel the launch, the link's 2 to 3 us and 256 KB at about 50 GB/s.  A model's input and output
// are [batch][features] on the host and [features][batch] in memory, so their kernels transpose (and pad) on the way, in
// pieces of columns that double from 128 KB on, instead of a transpose and a padding kernel each behind the copies: the same MLP
// 139 to 142 -> 129 to 135 us (at batch 2 / 4 / 16 54 / 67 / 69 -> 45 / 45 / 60, its narrow kernel included), 100-300-20 at batch 7 27 -> 20, the
// ResNet-18-shaped stack on 12 images of 96 x 96 490 -> 470.  One image (or sample) is the same in either order and goes as before.
constexpr size_t kStageIn = 4u << 20, kStageOut = 1u << 20, kStagePiece = 256u << 10, kStagePieceFirst = 128u << 10, kStagePieceMost = 1u << 20;
constexpr size_t kStageFlag = kStageIn + kStageOut;      // {turn, waits given up} behind the two areas
constexpr size_t kStagePairs = kStageFlag + 64;          // then the results that a launch writes itself: nothing else is ever there, so that an old pair has an old turn

// Words of up to two arrays, 16 bytes per thread and load (ends by the word).
__global__ __launch_bounds__(256)
void so_stage_in_kernel(uint32_t *dst, const uint32_t *src, uint32_t words, uint32_t *dst2, const uint32_t *src2, uint32_t words2)
{
    const uint32_t quads = words / 4u, quads2 = words2 / 4u, stride = gridDim.x * 256u;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < quads + quads2; i += stride) {
        if (i < quads) reinterpret_cast<uint4 *>(dst)[i] = reinterpret_cast<const uint4 *>(src)[i];
        else reinterpret_cast<uint4 *>(dst2)[i - quads] = reinterpret_cast<const uint4 *>(src2)[i - quads];
    }
    if (blockIdx.x != 0) return;
    if (threadIdx.x < words % 4u) dst[quads * 4u + threadIdx.x] = src[quads * 4u + threadIdx.x];
    if (threadIdx.x < words2 % 4u) dst2[quads2 * 4u + threadIdx.x] = src2[quads2 * 4u + threadIdx.x];
}

// dst[c * stride + r] = src[r * pitch + c] for the `rows` rows of a piece of `cols` columns, zeros for the rows up to `stride`: 64 columns
// by 32 rows per workgroup, 16 bytes per lane over the link (pitch is a multiple of four), 128 bytes at a time to memory.
__global__ __launch_bounds__(256)
void so_stage_in_transposed_kernel(float *dst, uint32_t stride, const float *src, uint32_t pitch, uint32_t rows, uint32_t cols)
{
    __shared__ float tile[64][33];
    const uint32_t r0 = blockIdx.y * 32u, c0 = blockIdx.x * 64u;
    const uint32_t c4 = (threadIdx.x & 15u) * 4u;
    float4 v[2];
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t r = r0 + k * 16u + (threadIdx.x >> 4);
        v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < rows && c0 + c4 < cols) v[k] = *reinterpret_cast<const float4 *>(src + (size_t)r * pitch + c0 + c4);
    }
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t r = k * 16u + (threadIdx.x >> 4);
        tile[c4][r] = v[k].x; tile[c4 + 1u][r] = v[k].y; tile[c4 + 2u][r] = v[k].z; tile[c4 + 3u][r] = v[k].w;
    }
    __syncthreads();
    const uint32_t r = threadIdx.x & 31u;
    for (uint32_t c = threadIdx.x >> 5; c < 64u; c += 8u)
        if (c0 + c < cols && r0 + r < stride) dst[(size_t)(c0 + c) * stride + r0 + r] = tile[c][r];
}

// The end of a way out: the last workgroup to finish tells the host: `turn`, and with it in one store the word of the bounded waits.  (A store
// for each and a fence between them: 0.6 us more of the encoder's 16 to 18 on small matrices, 0.7 of a model's 24.)
__device__ __forceinline__ void tell_host(uint32_t *done, const uint32_t *gave_up, uint32_t *flag, uint32_t turn)
{
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (gridDim.x > 1u) {
        if (__hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1u) return;
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(flag), (unsigned long long)*gave_up << 32 | turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// (Kernels of their own: one kernel for both, on a branch, cost each ellpack_matvec from host arrays 0.2 to 0.4 us of 18 to 20.)
__global__ __launch_bounds__(256)
void so_stage_out_kernel(uint32_t *dst, const uint32_t *src, uint32_t words, uint32_t *done, const uint32_t *gave_up, uint32_t *flag, uint32_t turn)
{
    const uint32_t quads = words / 4u, stride = gridDim.x * 256u;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < quads; i += stride) reinterpret_cast<uint4 *>(dst)[i] = reinterpret_cast<const uint4 *>(src)[i];
    if (blockIdx.x == 0 && threadIdx.x < words % 4u) dst[quads * 4u + threadIdx.x] = src[quads * 4u + threadIdx.x];
    tell_host(done, gave_up, flag, turn);
}

// dst is the transpose of src, whose rows of `cols` words lie `pitch` apart.
__global__ __launch_bounds__(256)
void so_stage_out_transposed_kernel(uint32_t *dst, const uint32_t *src, uint32_t words, uint32_t cols, uint32_t pitch, uint32_t *done, const uint32_t *gave_up, uint32_t *flag, uint32_t turn)
{
    const uint32_t quads = words / 4u, stride = gridDim.x * 256u, rows = words / cols;
    auto word = [&](uint32_t e) { const uint32_t c = e / rows; return src[(size_t)(e - c * rows) * pitch + c]; };
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < quads; i += stride)
        reinterpret_cast<uint4 *>(dst)[i] = make_uint4(word(4u * i), word(4u * i + 1u), word(4u * i + 2u), word(4u * i + 3u));
    if (blockIdx.x == 0 && threadIdx.x < words % 4u) dst[quads * 4u + threadIdx.x] = word(quads * 4u + threadIdx.x);
    tell_host(done, gave_up, flag, turn);
}

// A result of fewer than kStagePairsMost words as pairs {value, turn}, behind them the word of the bounded waits: what the host polls is the result itself, without
// a fence over the link and a word behind it.  cols != 0: a transpose, as above.  Models host to host, us, with the fence and the word / so: 85-351-177 at batch 5
// 20.5 / 18.5, 100-300-20 at 1 18.4 / 16.6, 100-300-1000 at 8 (8000 words) 22.8 / 20.9, 100-300-64 at 100 25.0 / 22.9.
__global__ __launch_bounds__(256)
void so_stage_pairs_kernel(uint2 *pairs, const uint32_t *src, uint32_t words, uint32_t cols, uint32_t pitch, const uint32_t *gave_up, uint32_t turn)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, rows = cols ? words / cols : 0u;
    if (i > words) return;
    uint32_t v;
    if (i == words) v = *gave_up;
    else if (cols == 0u) v = src[i];
    else {
        const uint32_t c = i / rows;
        v = src[(size_t)(i - c * rows) * pitch + c];
    }
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(pairs + i), (unsigned long long)turn << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The staging memory, made on first use.  False where there is none: the callers then copy as so_h2d and so_d2h do.
static bool stage_ready(so_ctx *ctx)
{
    if (ctx->h_stage) return true;
    void *p = nullptr, *d = nullptr;
    if (hipHostMalloc(&p, kStagePairs + kStagePairsMost * 8, hipHostMallocCoherent) != hipSuccess) { (void)hipGetLastError(); return false; }
    // cleared on the context's stream, which does not wait for the null stream
    if (hipMalloc(&d, 64) != hipSuccess || so_fill_zero(ctx, d, 64) != SO_OK) {
        (void)hipGetLastError();
        if (d) (void)hipFree(d);
        (void)hipHostFree(p);
        return false;
    }
    std::memset((char *)p + kStageFlag, 0, 64 + kStagePairsMost * 8);
    ctx->h_stage = (char *)p;
    ctx->d_stage_done = (uint32_t *)d;
    ctx->stage_used = 0;
    ctx->stage_turn = 0;
    return true;
}

extern "C" so_status so_stage_in(so_ctx *ctx, void *dst, const void *src, size_t bytes, void *dst2, const void *src2, size_t bytes2)
{
    SO_REQUIRE(ctx != nullptr, "so_stage_in: ctx is null");
    SO_REQUIRE((dst && src) || bytes == 0, "so_stage_in: null pointer");
    SO_REQUIRE((dst2 && src2) || bytes2 == 0, "so_stage_in: null pointer");
    SO_REQUIRE(!ctx->capturing, "so_stage_in: not allowed while a graph is being recorded");
    if (bytes + bytes2 == 0) return SO_OK;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const bool fits = bytes <= kStageIn && bytes2 <= kStageIn && ctx->stage_used + up(bytes) + up(bytes2) <= kStageIn;
    const bool aligned = bytes % 4 == 0 && bytes2 % 4 == 0 && ((uintptr_t)dst & 15) == 0 && ((uintptr_t)dst2 & 15) == 0;
    if (!fits || !aligned || !stage_ready(ctx)) {
        const so_status s = so_h2d(ctx, dst, src, bytes);
        return s != SO_OK ? s : so_h2d(ctx, dst2, src2, bytes2);
    }
    // the first array in pieces, the second with the last of them
    size_t at = 0;
    do {
        const size_t piece = std::min(kStagePiece, bytes - at);
        const bool last = at + piece == bytes;
        char *const h = ctx->h_stage + ctx->stage_used, *const h2 = h + up(piece);
        if (piece) std::memcpy(h, (const char *)src + at, piece);
        if (last && bytes2) std::memcpy(h2, src2, bytes2);
        const size_t both = piece + (last ? bytes2 : 0);
        const uint32_t blocks = (uint32_t)std::min<size_t>((both + 4095) / 4096, 256);
        so_stage_in_kernel<<<blocks, 256, 0, ctx->stream>>>((uint32_t *)((char *)dst + at), (const uint32_t *)h, (uint32_t)(piece / 4),
                                                            (uint32_t *)dst2, (const uint32_t *)h2, last ? (uint32_t)(bytes2 / 4) : 0u);
        SO_LAUNCH_CHECK();
        ctx->stage_used += up(piece) + (last ? up(bytes2) : 0);
        at += piece;
    } while (at < bytes);
    return SO_OK;
}

// Polls for `turn` in a word that the stream's last kernel writes.  *told: false where the stream ended without it; a stream
// that has failed ends the wait as well.
static so_status poll_word(so_ctx *ctx, volatile uint32_t *flag, uint32_t turn, bool *told)
{
    *told = true;
    for (uint32_t spin = 1; *flag != turn; ++spin) {
        if (spin % 4096u == 0) {
            const hipError_t e = hipStreamQuery(ctx->stream);
            if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
            SO_HIP(e);
            if (*flag != turn) { *told = false; return SO_OK; }
        }
        __builtin_ia32_pause();
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    ctx->stage_used = 0;                       // the stream's earlier work, and with it every way in, is done
    return SO_OK;
}

bool so_stage_result(so_ctx *ctx, uint32_t floats, uint2 **rows, uint32_t *turn)
{
    // (a launch with bounded waits before this one: the general way back looks at their word)
    if (floats > kStagePairsMost || ctx->waits_pending || !stage_ready(ctx)) return false;
    *rows = (uint2 *)(ctx->h_stage + kStagePairs);
    *turn = ++ctx->stage_turn;
    return true;
}

// The pairs from place `from` on, as their turn comes.
static so_status take_pairs(so_ctx *ctx, uint32_t from, uint32_t floats, const uint32_t *order, void *dst, uint32_t turn, bool *told)
{
    volatile const uint64_t *const rows = (volatile const uint64_t *)(ctx->h_stage + kStagePairs) + from;
    *told = true;
    uint32_t at = 0;
    for (uint32_t spin = 1; at < floats; ++spin) {
        for (uint64_t pair; at < floats && (uint32_t)((pair = rows[at]) >> 32) == turn; ++at) {
            const uint32_t bits = (uint32_t)pair;
            std::memcpy((char *)dst + 4 * (size_t)(order ? order[at] : at), &bits, 4);
        }
        if (at == floats) break;
        if (spin % 4096u == 0) {
            const hipError_t e = hipStreamQuery(ctx->stream);
            if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
            SO_HIP(e);
            if ((uint32_t)(rows[at] >> 32) != turn) { *told = false; return SO_OK; }
        }
        __builtin_ia32_pause();
    }
    ctx->stage_used = 0;                       // the stream's earlier work, and with it every way in, is done
    return SO_OK;
}

so_status so_stage_result_take(so_ctx *ctx, uint32_t floats, const uint32_t *order, float *dst, uint32_t turn, bool *told)
{
    return take_pairs(ctx, 0u, floats, order, dst, turn, told);
}

__global__ void so_tell_host_kernel(const uint32_t *gave_up, uint32_t *flag, uint32_t turn) { tell_host(nullptr, gave_up, flag, turn); }

// so_stream_wait by a kernel's word in the pinned memory that so_init made: that kernel starts when the stream's work before it is done
// and its results are where other streams see them.  The encoder's calls, us, hipStreamSynchronize / this: 256 x 256 19.7 / 17.7,
// 1024 x 1024 22.9 / 20.8, 4096 x 4096 36.5 / 34.8, 3738 x 7135 57.0 / 55.5; but 8192 x 8192, at 90 and 80 % sparse, 92.2 / 94.2 and 104.5 / 107.9:
// beyond kToldElements the extra launch costs what the earlier word gives.
constexpr uint64_t kToldElements = 1u << 25;
static so_status told_wait(so_ctx *ctx, uint64_t elements, const char *who)
{
    if (elements > kToldElements) return so_stream_wait(ctx, who);
    const so_tell tell = so_tell_next(ctx);
    so_tell_host_kernel<<<1, 64, 0, ctx->stream>>>(tell.gave_up, tell.flag, tell.turn);
    SO_LAUNCH_CHECK();
    return so_tell_wait(ctx, who);
}

so_tell so_tell_next(so_ctx *ctx)
{
    return so_tell{ctx->d_wait_gave_up, (uint32_t *)ctx->h_wait_gave_up + 12, ++ctx->told_turn};
}

so_status so_tell_wait(so_ctx *ctx, const char *who)
{
    volatile uint32_t *const flag = ctx->h_wait_gave_up + 12;
    bool told = false;
    const so_status s = poll_word(ctx, flag, ctx->told_turn, &told);
    if (s != SO_OK) return s;
    if (!told || (ctx->waits_pending && flag[1] != 0)) return so_stream_wait(ctx, who);
    ctx->waits_pending = false;
    return SO_OK;
}

// A copy of `bytes` (a transpose where cols != 0) to the staging memory, the wait for it, and from there to dst.  *told: false where the
// stream ended without the word.
static so_status stage_out(so_ctx *ctx, void *dst, const void *src, size_t bytes, uint32_t cols, uint32_t pitch, const char *who, bool *told)
{
    volatile uint32_t *const flag = (volatile uint32_t *)(ctx->h_stage + kStageFlag);
    const uint32_t turn = ++ctx->stage_turn;
    if (bytes / 4 < kStagePairsMost) {
        const uint32_t words = (uint32_t)(bytes / 4);
        so_stage_pairs_kernel<<<words / 256u + 1u, 256, 0, ctx->stream>>>((uint2 *)(ctx->h_stage + kStagePairs), (const uint32_t *)src, words, cols, pitch, ctx->d_wait_gave_up, turn);
        SO_LAUNCH_CHECK();
        uint32_t gave_up = 0;
        so_status s = ctx->waits_pending ? take_pairs(ctx, words, 1u, nullptr, &gave_up, turn, told) : SO_OK;
        if (s == SO_OK && gave_up != 0) return so_stream_wait(ctx, who);
        if (s == SO_OK && (!ctx->waits_pending || *told)) s = take_pairs(ctx, 0u, words, nullptr, dst, turn, told);
        if (s == SO_OK && *told) ctx->waits_pending = false;
        return s;
    }
    const uint32_t blocks = (uint32_t)std::min<size_t>((bytes + 8191) / 8192, 128);
    uint32_t *const to = (uint32_t *)(ctx->h_stage + kStageIn);
    if (cols == 0)
        so_stage_out_kernel<<<blocks, 256, 0, ctx->stream>>>(to, (const uint32_t *)src, (uint32_t)(bytes / 4), ctx->d_stage_done, ctx->d_wait_gave_up, (uint32_t *)flag, turn);
    else
        so_stage_out_transposed_kernel<<<blocks, 256, 0, ctx->stream>>>(to, (const uint32_t *)src, (uint32_t)(bytes / 4), cols, pitch,
                                                                        ctx->d_stage_done, ctx->d_wait_gave_up, (uint32_t *)flag, turn);
    SO_LAUNCH_CHECK();
    const so_status s = poll_word(ctx, flag, turn, told);
    if (s != SO_OK || !*told) return s;
    if (ctx->waits_pending && flag[1] != 0) return so_stream_wait(ctx, who);
    ctx->waits_pending = false;
    std::memcpy(dst, ctx->h_stage + kStageIn, bytes);
    return SO_OK;
}

extern "C" so_status so_stage_out(so_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    SO_REQUIRE(ctx != nullptr, "so_stage_out: ctx is null");
    if (bytes == 0) return SO_OK;
    SO_REQUIRE(dst && src, "so_stage_out: null pointer");
    SO_REQUIRE(!ctx->capturing, "so_stage_out: not allowed while a graph is being recorded");
    if (bytes > kStageOut || bytes % 4 != 0 || ((uintptr_t)src & 15) != 0 || !stage_ready(ctx)) return so_d2h(ctx, dst, src, bytes);
    bool told = false;
    const so_status s = stage_out(ctx, dst, src, bytes, 0u, 0u, "so_stage_out", &told);
    return s != SO_OK || told ? s : so_d2h(ctx, dst, src, bytes);
}

extern "C" so_status so_stage_in_transposed(so_ctx *ctx, float *dDst, uint32_t stride, const float *src, uint32_t rows, uint32_t cols, int *done)
{
    SO_REQUIRE(ctx && done, "so_stage_in_transposed: null argument");
    *done = 1;
    if (rows == 0 || cols == 0) return SO_OK;
    SO_REQUIRE(dDst && src, "so_stage_in_transposed: null pointer");
    SO_REQUIRE(stride >= rows, "so_stage_in_transposed: %u values a row, %u rows", stride, rows);
    SO_REQUIRE(!ctx->capturing, "so_stage_in_transposed: not allowed while a graph is being recorded");
    // All pieces but the last are of whole 256 bytes a row.  Rows: host to memory, this way and staged with a transpose behind it, us:
    // 3000 x 10 18.9 / 22.5, 4000 x 64 50.7 / 52.0, 4100 x 250 127 / 145, 8000 x 80 108 / 99, 8000 x 4 24.8 / 21.4; 1000 x 1 16.0 / 17.5, 3000 x 1 19.0 / 17.3.
    const size_t row_bytes = ((size_t)cols + 3) / 4 * 16, want = row_bytes * rows + 255;
    const bool pays = rows <= 1024u * std::min(cols, 4u);
    if (!pays || want > kStageIn || ctx->stage_used + want > kStageIn || so_ceil_div(stride, 32) > 65535u || !stage_ready(ctx)) { *done = 0; return SO_OK; }
    // pieces of columns: the first small, so that the link starts early, each of the others twice the one before it
    size_t piece = kStagePieceFirst;
    for (uint32_t at = 0; at < cols; piece = std::min(2 * piece, kStagePieceMost)) {
        const uint32_t n = (uint32_t)std::min<size_t>(cols - at, std::max<size_t>(64, piece / (4 * (size_t)rows) / 64 * 64)), pitch = (n + 3u) / 4u * 4u;
        float *const h = (float *)(ctx->h_stage + ctx->stage_used);
        for (uint32_t r = 0; r < rows; ++r) std::memcpy(h + (size_t)r * pitch, src + (size_t)r * cols + at, (size_t)n * 4);
        so_stage_in_transposed_kernel<<<dim3(so_ceil_div(n, 64), so_ceil_div(stride, 32)), 256, 0, ctx->stream>>>(dDst + (size_t)at * stride, stride, h, pitch, rows, n);
        SO_LAUNCH_CHECK();
        ctx->stage_used += ((size_t)rows * pitch * 4 + 255) / 256 * 256;
        at += n;
    }
    return SO_OK;
}

extern "C" so_status so_stage_out_transposed(so_ctx *ctx, float *dst, const float *dSrc, uint32_t stride, uint32_t rows, uint32_t cols, int *done)
{
    SO_REQUIRE(ctx && done, "so_stage_out_transposed: null argument");
    *done = 1;
    if (rows == 0 || cols == 0) return SO_OK;
    SO_REQUIRE(dst && dSrc, "so_stage_out_transposed: null pointer");
    SO_REQUIRE(stride >= cols, "so_stage_out_transposed: %u values a row, %u columns", stride, cols);
    SO_REQUIRE(!ctx->capturing, "so_stage_out_transposed: not allowed while a graph is being recorded");
    *done = 0;
    if ((uint64_t)rows * cols * 4 > kStageOut || !stage_ready(ctx)) return SO_OK;
    bool told = false;
    const so_status s = stage_out(ctx, dst, dSrc, (size_t)rows * cols * 4, cols, stride, "so_stage_out_transposed", &told);
    *done = told;
    return s;
}

extern "C" so_status so_d2d(so_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    SO_REQUIRE(ctx != nullptr, "so_d2d: ctx is null");
    if (bytes == 0) return SO_OK;
    SO_REQUIRE(dst && src, "so_d2d: null pointer");
    SO_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    return SO_OK;
}

__global__ void so_fill_zero_kernel(uint32_t *p, size_t words)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < words; i += stride) p[i] = 0u;
}

extern "C" so_status so_fill_zero(so_ctx *ctx, void *dptr, size_t bytes)
{
    SO_REQUIRE(ctx != nullptr, "so_fill_zero: ctx is null");
    if (bytes == 0) return SO_OK;
    SO_REQUIRE(dptr != nullptr && bytes % 4 == 0 && ((uintptr_t)dptr & 3) == 0,
               "so_fill_zero: pointer and size must be 4-byte multiples");
    const size_t words = bytes / 4;
    const uint32_t blocks = (uint32_t)std::min<size_t>((words + 255) / 256, 4096);
    so_fill_zero_kernel<<<blocks, 256, 0, ctx->stream>>>((uint32_t *)dptr, words);
    SO_LAUNCH_CHECK();
    return SO_OK;
}

extern "C" so_status so_sync(so_ctx *ctx)
{
    SO_REQUIRE(ctx != nullptr, "so_sync: ctx is null");
    SO_REQUIRE(!ctx->capturing, "so_sync: not allowed while a graph is being recorded");
    // a kernel whose waves gave up waiting for one another has produced garbage: say so
    return so_stream_wait(ctx, "so_sync");
}

extern "C" so_status so_timer_begin(so_ctx *ctx)
{
    SO_REQUIRE(ctx != nullptr, "so_timer_begin: ctx is null");
    SO_REQUIRE(!ctx->capturing, "so_timer_begin: not allowed while a graph is being recorded");
    SO_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    return SO_OK;
}

extern "C" so_status so_timer_end(so_ctx *ctx, float *ms)
{
    SO_REQUIRE(ctx && ms, "so_timer_end: null argument");
    SO_REQUIRE(!ctx->capturing, "so_timer_end: not allowed while a graph is being recorded");
    SO_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    const so_status s = so_stream_wait(ctx, "so_timer_end");
    SO_HIP(hipEventElapsedTime(ms, ctx->ev0, ctx->ev1));
    return s;
}

// ---------------------------------------------------------------- launch graphs

extern "C" so_status so_graph_begin(so_ctx *ctx)
{
    SO_REQUIRE(ctx != nullptr, "so_graph_begin: ctx is null");
    SO_REQUIRE(!ctx->capturing, "so_graph_begin: already recording");
    SO_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    ctx->capturing = true;
    return SO_OK;
}

extern "C" so_status so_graph_end(so_ctx *ctx, so_graph **out)
{
    SO_REQUIRE(ctx && out, "so_graph_end: null argument");
    SO_REQUIRE(ctx->capturing, "so_graph_end: not recording");
    *out = nullptr;
    ctx->capturing = false;
    std::vector<so_block_ref> uses = std::move(ctx->recorded);
    ctx->recorded.clear();
    hipGraph_t graph = nullptr;
    SO_HIP(hipStreamEndCapture(ctx->stream, &graph));
    so_graph *g = new (std::nothrow) so_graph();
    if (!g) { (void)hipGraphDestroy(graph); so_set_error("so_graph_end: host allocation failed"); return SO_ERR_OOM; }
    g->graph = graph;
    g->uses = std::move(uses);
    hipError_t e = hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        so_set_error("hipGraphInstantiate failed: %s", hipGetErrorString(e));
        (void)hipGraphDestroy(graph);
        delete g;
        return SO_ERR_HIP;
    }
    *out = g;
    return SO_OK;
}

extern "C" so_status so_graph_launch(so_ctx *ctx, so_graph *g)
{
    SO_REQUIRE(ctx && g && g->exec, "so_graph_launch: null argument");
    SO_REQUIRE(!ctx->capturing, "so_graph_launch: not allowed while recording");
    SO_HIP(hipGraphLaunch(g->exec, ctx->stream));
    ctx->waits_pending = true;          // the graph may hold kernels with bounded waits
    return SO_OK;
}

extern "C" so_status so_graph_free(so_ctx *ctx, so_graph *g)
{
    if (!g) return SO_OK;
    if (ctx && ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return SO_OK;
}

// ------------------------------------------------------------ ELLPACK on device

static void free_ellpack_arrays(so_ellpack *E)
{
    if (E->d_Wd) (void)hipFree(E->d_Wd);
    if (E->d_idx) (void)hipFree(E->d_idx);
    if (E->d_nnz) (void)hipFree(E->d_nnz);
    if (E->d_WdT) (void)hipFree(E->d_WdT);
    if (E->d_idxT) (void)hipFree(E->d_idxT);
    if (E->d_idx16) (void)hipFree(E->d_idx16);
    if (E->d_idxT16) (void)hipFree(E->d_idxT16);
    for (auto &b : E->bins)
        if (b.d_rows) (void)hipFree(b.d_rows);
    if (E->tiled.d_entries) (void)hipFree(E->tiled.d_entries);
    if (E->tiled.d_info) (void)hipFree(E->tiled.d_info);
    if (E->tiled.d_rows) (void)hipFree(E->tiled.d_rows);
    so_rbmm_free(E);
    so_planes_free(E);
    so_quads_free(E);
}

// Device copy of a host array with 16 zeroed bytes after the last element, so a
// kernel may read whole aligned 16-byte groups that straddle the end.
template <typename T>
static so_status upload_array(so_ctx *ctx, const T *host, size_t count, T **dev)
{
    void *p = nullptr;
    so_status s = so_malloc(ctx, count * sizeof(T) + 16, &p);
    if (s != SO_OK) return s;
    *dev = (T *)p;
    SO_HIP(hipMemsetAsync((char *)p + count * sizeof(T), 0, 16, ctx->stream));
    return so_h2d(ctx, p, host, count * sizeof(T));
}

// K-tiled layout for the LDS-staged matmul (see so_tiled).  Rows are first ordered
// by stored-nonzero count (longest first, stable; over the whole matrix or inside
// each workgroup's block of 64 rows, see below) so that the four rows sharing a
// wavefront have similar lengths; the order only decides which rows share a wave,
// every row is still written to its own place in Y.
static so_status build_tiled(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz)
{
    const uint32_t m = E->m, n = E->n, r = E->r;
    constexpr uint32_t KT = so_tiled::kTileRows, ROWB = so_tiled::kSlabCols * 4;
    so_tiled &T = E->tiled;
    T.nquads = (m + 3) / 4;
    T.ntiles = std::max(1u, (n + KT - 1) / KT);
    // Two candidate orders: sorted by length over the whole matrix, or only inside blocks of 64
    // consecutive rows (the rows of one workgroup).  The second keeps a workgroup's rows of Y next
    // to each other, which is worth ~5 % of a launch; the first is needed when lengths vary so
    // much that rows of one block do not fit together.  Take the block-wise order unless the
    // global one saves more than 2 % of the steps.
    const auto longer_first = [&](uint32_t a, uint32_t b) { return nnz[a] > nnz[b]; };
    std::vector<uint32_t> order(m), blockwise(m);
    for (uint32_t i = 0; i < m; ++i) order[i] = blockwise[i] = i;
    std::stable_sort(order.begin(), order.end(), longer_first);
    for (uint32_t b0 = 0; b0 < m; b0 += 64)
        std::stable_sort(blockwise.begin() + b0, blockwise.begin() + std::min(m, b0 + 64), longer_first);
    if ((uint64_t)m * T.ntiles <= (1ull << 28)) {                     // the comparison needs 2 bytes per (row, tile)
        std::vector<uint16_t> per_tile((size_t)m * T.ntiles, 0);      // a tile has at most 256 columns
        so_parallel(m, E->total_nnz, [&](uint32_t i0, uint32_t i1) {
            for (uint32_t i = i0; i < i1; ++i)
                for (uint32_t k = 0; k < nnz[i]; ++k) ++per_tile[(size_t)i * T.ntiles + idx[(size_t)i * r + k] / KT];
        });
        const auto steps_of = [&](const std::vector<uint32_t> &ord) {
            uint64_t total = 0;
            for (uint32_t q0 = 0; q0 < m; q0 += 4)
                for (uint32_t t = 0; t < T.ntiles; ++t) {
                    uint32_t most = 0;
                    for (uint32_t g = q0; g < std::min(m, q0 + 4); ++g) most = std::max<uint32_t>(most, per_tile[(size_t)ord[g] * T.ntiles + t]);
                    total += (most + 3u) & ~3u;
                }
            return total;
        };
        if (steps_of(blockwise) * 100 <= steps_of(order) * 102) order.swap(blockwise);
    }
    std::vector<uint32_t> qrows((size_t)T.nquads * 4, 0xffffffffu);
    for (uint32_t i = 0; i < m; ++i) qrows[i] = order[i];

    // Steps per (quad, tile) first, then every quad fills in its own chunks.
    std::vector<so_tile_info> info((size_t)T.nquads * T.ntiles);
    const auto walk = [&](uint32_t q, const auto &tile) {             // tile(t, first slot of each row in tile t, slots)
        uint32_t pos[4] = {0, 0, 0, 0};
        for (uint32_t t = 0; t < T.ntiles; ++t) {
            const uint64_t col_end = (uint64_t)(t + 1) * KT;
            uint32_t cnt[4] = {0, 0, 0, 0};
            for (int g = 0; g < 4; ++g) {
                const uint32_t row = qrows[(size_t)q * 4 + g];
                if (row == 0xffffffffu) continue;
                const uint32_t *c = idx + (size_t)row * r;
                uint32_t p = pos[g];
                while (p < nnz[row] && c[p] < col_end) ++p;
                cnt[g] = p - pos[g];
            }
            tile(t, pos, cnt);
            for (int g = 0; g < 4; ++g) pos[g] += cnt[g];
        }
    };
    so_parallel(T.nquads, E->total_nnz, [&](uint32_t q0, uint32_t q1) {
        for (uint32_t q = q0; q < q1; ++q)
            walk(q, [&](uint32_t t, const uint32_t *, const uint32_t *cnt) {
                info[(size_t)q * T.ntiles + t].steps = (std::max(std::max(cnt[0], cnt[1]), std::max(cnt[2], cnt[3])) + 3u) & ~3u;
            });
    });
    uint64_t total_steps = 0, chunks = 0;
    for (so_tile_info &i : info) {
        if (chunks > 0xfffffff0ull) { so_set_error("so_ellpack_upload: matrix too large for the tiled layout"); return SO_ERR_INVALID; }
        i.chunk0 = (uint32_t)chunks;
        chunks += (i.steps + 15) / 16;
        total_steps += i.steps;
    }
    std::vector<so_tile_entry> entries((size_t)chunks * 64);
    so_parallel(T.nquads, E->total_nnz, [&](uint32_t q0, uint32_t q1) {
        for (uint32_t q = q0; q < q1; ++q)
            walk(q, [&](uint32_t t, const uint32_t *pos, const uint32_t *cnt) {
                // The zero row sits after both tile buffers; offsets are relative to the buffer the tile uses.
                // A padding step is fma(-0, +0, acc): adding -0 leaves every accumulator, -0 included, as it is.
                const uint32_t zero_off = so_tiled::kZeroRowOff - (t & 1u) * so_tiled::kTileBytes;
                const so_tile_info &in = info[(size_t)q * T.ntiles + t];
                so_tile_entry *out = entries.data() + (size_t)in.chunk0 * 64;
                for (uint32_t ch = 0; ch < (in.steps + 15) / 16; ++ch)
                    for (int g = 0; g < 4; ++g)
                        for (uint32_t k = 0; k < 16; ++k) {
                            const uint32_t sidx = ch * 16 + k;
                            so_tile_entry e{-0.0f, zero_off};
                            if (sidx < cnt[g]) {
                                const size_t slot = (size_t)qrows[(size_t)q * 4 + g] * r + pos[g] + sidx;
                                e.w = Wd[slot];
                                e.off = (idx[slot] - t * KT) * ROWB;
                            }
                            *out++ = e;
                        }
            });
    });
    // Three zero chunks of slack: the kernel always fetches three chunks per tile.
    entries.resize(entries.size() + 3 * 64, so_tile_entry{-0.0f, so_tiled::kZeroRowOff});
    T.total_steps = total_steps;
    so_status s = upload_array(ctx, entries.data(), entries.size(), &T.d_entries);
    if (s == SO_OK) s = upload_array(ctx, info.data(), info.size(), &T.d_info);
    if (s == SO_OK) s = upload_array(ctx, qrows.data(), qrows.size(), &T.d_rows);
    return s;
}

extern "C" so_status so_ellpack_upload(so_ctx *ctx, const float *Wd, const uint32_t *idx,
                                       const uint32_t *nnz, uint32_t m, uint32_t n, uint32_t r,
                                       int layouts, so_ellpack **out)
{
    SO_REQUIRE(ctx && out, "so_ellpack_upload: null argument");
    *out = nullptr;
    const size_t slots = (size_t)m * r;
    SO_REQUIRE(m == 0 || nnz != nullptr, "so_ellpack_upload: nnz is null");
    SO_REQUIRE(slots == 0 || (Wd && idx), "so_ellpack_upload: Wd/idx is null");
    SO_REQUIRE((layouts & ~(SO_LAYOUT_ROW | SO_LAYOUT_SLOT | SO_LAYOUT_BINS | SO_LAYOUT_TILED | SO_LAYOUT_RBM | SO_LAYOUT_IDX16)) == 0,
               "so_ellpack_upload: unknown layout bits 0x%x", layouts);
    SO_REQUIRE(!(layouts & SO_LAYOUT_IDX16) || n <= 65536u, "so_ellpack_upload: 16-bit columns need n <= 65536 (n = %u)", n);

    // Validate on the host before anything reaches a kernel: every stored slot must
    // name a column inside X, every count must fit the row.
    // The encoder stores a row's columns in strictly ascending order and the K-tiled matmul layout
    // and the convolution's windowed layout walk a row on that assumption; a matrix filled in by
    // hand in any other order (the reference's kernels take slots in whatever order they come) is
    // served by the kernels that do the same, and the ordered layouts are not built for it.
    uint64_t total = 0;
    uint32_t max_nnz = 0;
    bool ascending = true;
    for (uint32_t i = 0; i < m; ++i) {
        const uint32_t c = nnz[i];
        if (c > r) {
            so_set_error("so_ellpack_upload: nnz[%u] = %u exceeds r = %u", i, c, r);
            return SO_ERR_BOUNDS;
        }
        const uint32_t *row = idx + (size_t)i * r;
        for (uint32_t k = 0; k < c; ++k) {
            if (row[k] >= n) {
                so_set_error("so_ellpack_upload: idx[%u,%u] = %u is not below n = %u", i, k, row[k], n);
                return SO_ERR_BOUNDS;
            }
            if (k > 0 && row[k] <= row[k - 1]) ascending = false;
        }
        total += c;
        max_nnz = std::max(max_nnz, c);
    }

    so_ellpack *E = new (std::nothrow) so_ellpack();
    if (!E) { so_set_error("so_ellpack_upload: host allocation failed"); return SO_ERR_OOM; }
    E->m = m; E->n = n; E->r = r;
    E->total_nnz = total;
    E->max_nnz = max_nnz;
    E->ascending = ascending;
    if (!ascending) layouts &= ~SO_LAYOUT_TILED;
    E->layouts = layouts | SO_LAYOUT_ROW;

    so_status s = SO_OK;
    try {
        s = upload_array(ctx, Wd, slots, &E->d_Wd);
        if (s == SO_OK) s = upload_array(ctx, idx, slots, &E->d_idx);
        if (s == SO_OK) s = upload_array(ctx, nnz, (size_t)m, &E->d_nnz);

        if (s == SO_OK && (layouts & SO_LAYOUT_SLOT)) {
            std::vector<float> WdT(slots);
            std::vector<uint32_t> idxT(slots);
            for (uint32_t i = 0; i < m; ++i)
                for (uint32_t k = 0; k < r; ++k) {
                    WdT[(size_t)k * m + i] = Wd[(size_t)i * r + k];
                    idxT[(size_t)k * m + i] = idx[(size_t)i * r + k];
                }
            s = upload_array(ctx, WdT.data(), slots, &E->d_WdT);
            if (s == SO_OK) s = upload_array(ctx, idxT.data(), slots, &E->d_idxT);
            if (s == SO_OK && (layouts & SO_LAYOUT_IDX16)) {
                std::vector<uint16_t> idxT16(slots);
                for (size_t k = 0; k < slots; ++k) idxT16[k] = (uint16_t)idxT[k];
                s = upload_array(ctx, idxT16.data(), slots, &E->d_idxT16);
            }
        }

        if (s == SO_OK && (layouts & SO_LAYOUT_IDX16)) {
            // The same slots as d_idx, two bytes each: so_matvec streams 6 bytes per nonzero instead of 8.
            // Padding slots keep the low half of whatever they hold; no kernel uses them.
            std::vector<uint16_t> idx16(slots);
            for (size_t k = 0; k < slots; ++k) idx16[k] = (uint16_t)idx[k];
            s = upload_array(ctx, idx16.data(), slots, &E->d_idx16);
        }

        if (s == SO_OK && (layouts & SO_LAYOUT_BINS)) {
            // Length classes: <= 16 nonzeros -> 4 lanes per row, <= 128 -> 16 lanes, <= 4096 -> a whole
            // wave, longer -> a whole workgroup (a single wave would walk such a row long after every
            // other row is done).  Long rows first inside a class, so the last waves to start are the
            // short ones.
            static const uint32_t group[4] = {4, 16, 64, 1024};
            static const uint32_t limit[4] = {16, 128, 4096, 0xffffffffu};
            std::vector<uint32_t> rows[4];
            for (uint32_t i = 0; i < m; ++i) {
                int b = 0;
                while (nnz[i] > limit[b]) ++b;
                rows[b].push_back(i);
            }
            for (int b = 0; b < 4 && s == SO_OK; ++b) {
                std::stable_sort(rows[b].begin(), rows[b].end(),
                                 [&](uint32_t a, uint32_t c) { return nnz[a] > nnz[c]; });
                E->bins[b].group = group[b];
                E->bins[b].count = (uint32_t)rows[b].size();
                // (row, its length) pairs: a wave learns where its row is and how long in one load
                std::vector<uint32_t> pairs(2 * rows[b].size());
                for (size_t k = 0; k < rows[b].size(); ++k) {
                    pairs[2 * k] = rows[b][k];
                    pairs[2 * k + 1] = nnz[rows[b][k]];
                }
                if (!pairs.empty()) s = upload_array(ctx, pairs.data(), pairs.size(), &E->bins[b].d_rows);
            }
            if (m <= kStagePairsMost)
                for (int b = 3; b >= 0; --b) E->bin_order.insert(E->bin_order.end(), rows[b].begin(), rows[b].end());
        }

        if (s == SO_OK && (layouts & SO_LAYOUT_TILED) && m > 0) s = build_tiled(ctx, E, Wd, idx, nnz);
        if (s == SO_OK && (layouts & SO_LAYOUT_RBM) && m > 0) s = so_rbmm_build(ctx, E, Wd, idx, nnz);
        if (s == SO_OK && (layouts & SO_LAYOUT_RBM) && m > 0) {
            // the layout's second copy: where there is no memory for it the handle does without
            try {
                s = so_quads_build(ctx, E, Wd, idx, nnz);
            } catch (const std::bad_alloc &) {
                s = SO_ERR_OOM;
            }
            if (s == SO_ERR_OOM) { (void)hipGetLastError(); so_quads_free(E); s = SO_OK; }
            // and a third where the matrix is full enough
            if (s == SO_OK && so_planes_pays(ctx, E)) s = so_planes_build(ctx, E, Wd, nnz);
            if (s == SO_ERR_OOM) { (void)hipGetLastError(); so_planes_free(E); s = SO_OK; }
        }
    } catch (const std::exception &e) {                  // a builder ran out of host memory, on whichever thread
        so_set_error("so_ellpack_upload: building the layouts failed: %s", e.what());
        s = SO_ERR_OOM;
    }

    if (s != SO_OK) {
        free_ellpack_arrays(E);
        delete E;
        return s;
    }
    *out = E;
    return SO_OK;
}

extern "C" so_status so_ellpack_free(so_ctx *ctx, so_ellpack *E)
{
    if (!E) return SO_OK;
    if (ctx && ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    free_ellpack_arrays(E);
    delete E;
    return SO_OK;
}

extern "C" so_status so_ellpack_dims(const so_ellpack *E, uint32_t *m, uint32_t *n, uint32_t *r,
                                     uint64_t *total_nnz, int *layouts)
{
    SO_REQUIRE(E != nullptr, "so_ellpack_dims: E is null");
    if (m) *m = E->m;
    if (n) *n = E->n;
    if (r) *r = E->r;
    if (total_nnz) *total_nnz = E->total_nnz;
    if (layouts) *layouts = E->layouts;
    return SO_OK;
}

namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // rows of a dense matrix start anywhere

// Decoding: a workgroup builds up to kDecodeSpan consecutive elements of W in LDS -- whole rows, or a part of one longer
// row -- and writes them out once, 16 bytes per lane, past the caches (nontemporal: a plain store of W takes twice as
// long and pushes the matrix out of the Infinity Cache).
// Bound by the write of W: 8192 x 8192, 90 % sparse, 50 us (6.4 TB/s of its 322 MB), 80 on buffers not used before;
// 143 and 114 as a fill of W followed by a scatter of single words into it.  Without the requests ahead the chain
// length -> slots -> span -> write made it 67 and 140.
constexpr uint32_t kDecodeSpan = 8192;       // 32 KB: five workgroups per compute unit
constexpr uint32_t kDecodeSlots = 8;         // slots a thread has in registers

// Several rows per span, a wave takes every fourth.  The span starts as zeros and is put back to zeros after each use by
// clearing what was scattered.
__global__ __launch_bounds__(256)
void ellpack_decode_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx,
                           const uint32_t *__restrict__ nnz, uint32_t m, uint32_t n, uint32_t r,
                           float *__restrict__ W, uint32_t rows_per_span, uint32_t spans)
{
    __shared__ __attribute__((aligned(16))) float span[kDecodeSpan];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    f32x4u *span4 = reinterpret_cast<f32x4u *>(span);
    for (uint32_t k = tid; k < kDecodeSpan / 4u; k += 256u) *reinterpret_cast<float4 *>(span + 4u * k) = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t sp = blockIdx.x; sp < spans; sp += gridDim.x) {
        const uint32_t row0 = sp * rows_per_span, rows = min(rows_per_span, m - row0), count = rows * n;
        float *out = W + (size_t)row0 * n;
        auto scatter = [&](bool value) {               // false: the same places back to zero
            for (uint32_t i = wave; i < rows; i += 4u) {
                const uint32_t c = nnz[row0 + i];
                const uint32_t *ix = idx + (size_t)(row0 + i) * r;
                const float *wd = Wd + (size_t)(row0 + i) * r;
                for (uint32_t from = lane; from < c; from += kDecodeSlots * 64u) {
                    uint32_t at[kDecodeSlots];
                    float v[kDecodeSlots];
#pragma unroll
                    for (uint32_t u = 0; u < kDecodeSlots; ++u)
                        if (from + u * 64u < c) { at[u] = ix[from + u * 64u]; v[u] = wd[from + u * 64u]; }
#pragma unroll
                    for (uint32_t u = 0; u < kDecodeSlots; ++u)
                        if (from + u * 64u < c) span[i * n + at[u]] = value ? v[u] : 0.0f;
                }
            }
        };
        __syncthreads();                               // the span is all zeros
        scatter(true);
        __syncthreads();
        for (uint32_t k = tid; k < count / 4u; k += 256u) __builtin_nontemporal_store(span4[k], reinterpret_cast<f32x4u *>(out) + k);
        if (tid < (count & 3u)) out[(count & ~3u) + tid] = span[(count & ~3u) + tid];
        __syncthreads();
        scatter(false);
    }
}

// A span is (part of) one row; a work item is one of the row's `segs` shares of `per_seg` spans of `width` columns.  The
// row's slots come in batches of 2048 (eight per thread), the next batch -- of this row, else the next item's first -- on
// its way while this one is scattered and the span is written out.  Where the columns ascend (SORTED) a batch that reaches
// past the span is kept for the next one, so every slot is read once however many spans the row has; else each span
// goes through the whole row.  1024 x 65536, half full: 537 us with the whole row for each span, 360 as a fill and a
// scatter, 104 so; 10 % full 132, 145 and 53; 64 x 262144, 10 % full 61, 155 and 19.
template <bool SORTED>
__global__ __launch_bounds__(256)
void ellpack_decode_wide_kernel(const float *__restrict__ Wd, const uint32_t *__restrict__ idx, const uint32_t *__restrict__ nnz,
                                uint32_t n, uint32_t r, float *__restrict__ W, uint32_t width, uint32_t per_seg, uint32_t segs, uint32_t items)
{
    constexpr uint32_t kBatch = kDecodeSlots * 256u;
    __shared__ __attribute__((aligned(16))) float span[kDecodeSpan];
    const uint32_t tid = threadIdx.x;
    f32x4u *span4 = reinterpret_cast<f32x4u *>(span);
    for (uint32_t k = tid; k < kDecodeSpan / 4u; k += 256u) *reinterpret_cast<float4 *>(span + 4u * k) = make_float4(0.f, 0.f, 0.f, 0.f);

    struct Batch { uint32_t at[kDecodeSlots], last; float v[kDecodeSlots]; };      // columns (0xffffffff: no such slot), the last slot's among them, values
    auto request = [&](uint32_t row, uint32_t from, uint32_t cnt, Batch &b) {
        const uint32_t *ix = idx + (size_t)row * r;
        const float *wd = Wd + (size_t)row * r;
#pragma unroll
        for (uint32_t u = 0; u < kDecodeSlots; ++u) {
            const uint32_t k = from + tid + u * 256u;
            b.at[u] = 0xffffffffu;
            if (k < cnt) { b.at[u] = ix[k]; b.v[u] = wd[k]; }
        }
        if (SORTED && from + kBatch < cnt) b.last = ix[from + kBatch - 1u];        // only looked at when the row goes on
    };
    // SORTED: the row's first slot with a column of `col` or more
    auto first_slot = [&](uint32_t row, uint32_t col, uint32_t cnt) {
        const uint32_t *ix = idx + (size_t)row * r;
        uint32_t lo = 0, hi = cnt;
        while (lo < hi) {
            const uint32_t step = (hi - lo + 255u) / 256u, k = lo + tid * step;
            const uint32_t below = (uint32_t)__syncthreads_count(k < hi && ix[k] < col);
            hi = min(hi, lo + below * step);
            lo = below == 0u ? lo : lo + (below - 1u) * step + 1u;
        }
        return lo;
    };
    Batch cur, nxt;
    uint32_t item = blockIdx.x, row, col, col_end, cnt, from, cnt_next = 0, cnt_after = 0;      // cnt_next, cnt_after: rows of the two items to come (segs = 1)
    const uint32_t stride = gridDim.x;
    auto place = [&] {
        row = item / segs;
        col = (item - row * segs) * per_seg * width;
        col_end = (uint32_t)min((uint64_t)n, (uint64_t)col + (uint64_t)per_seg * width);
    };
    auto look_ahead = [&] {              // what follows the batch in `cur`
        if (from + kBatch < cnt) request(row, from + kBatch, cnt, nxt);
        else if (segs == 1u && item + stride < items) request(item + stride, 0, cnt_next, nxt);
    };
    place();
    cnt = nnz[row];
    from = SORTED && segs > 1u ? first_slot(row, col, cnt) : 0u;
    request(row, from, cnt, cur);
    if (segs == 1u && item + stride < items) cnt_next = nnz[item + stride];
    look_ahead();
    if (segs == 1u && item + 2u * stride < items) cnt_after = nnz[item + 2u * stride];
    for (;;) {
        for (;; col += width) {
            const uint32_t count = min(width, n - col);
            __syncthreads();                               // the span is all zeros
            for (;;) {
#pragma unroll
                for (uint32_t u = 0; u < kDecodeSlots; ++u) {
                    const uint32_t c = cur.at[u] - col;
                    if (cur.at[u] != 0xffffffffu && c < count) span[c] = cur.v[u];
                }
                if (from + kBatch >= cnt || (SORTED && cur.last >= col + count)) break;
                cur = nxt;
                from += kBatch;
                look_ahead();
            }
            __syncthreads();
            float *out = W + (size_t)row * n + col;
            for (uint32_t k = tid; k < count / 4u; k += 256u) {
                __builtin_nontemporal_store(span4[k], reinterpret_cast<f32x4u *>(out) + k);
                span4[k] = f32x4u{0.f, 0.f, 0.f, 0.f};
            }
            if (tid < (count & 3u)) {
                out[(count & ~3u) + tid] = span[(count & ~3u) + tid];
                span[(count & ~3u) + tid] = 0.0f;
            }
            if (col_end - col <= width) break;
            if (!SORTED && from != 0u) {                   // from the row's start again
                from = 0;
                request(row, 0, cnt, cur);
                look_ahead();
            }
        }
        item += stride;
        if (item >= items) break;
        place();
        if (segs == 1u) {
            cur = nxt;
            cnt = cnt_next;
            cnt_next = cnt_after;
            from = 0;
        } else {
            cnt = nnz[row];
            from = SORTED ? first_slot(row, col, cnt) : 0u;
            request(row, from, cnt, cur);
        }
        look_ahead();
        if (segs == 1u && item + 2u * stride < items) cnt_after = nnz[item + 2u * stride];
    }
}

} // namespace

namespace {

// The encoder's counting pass leaves one partial result per workgroup -- the longest row and the
// number of nonzeros among the workgroup's rows -- in a scratch buffer; the packing pass folds them
// (each workgroup for itself up to kEncodeFoldBlocks of them; beyond, a one-workgroup pass does it once)
// into {r, total nnz}, so the row pitch of the output never travels through the host.
// Layout of the scratch buffer: header {r, total nnz (low, high), 0} (kEncodeHeaderBytes), then one uint2
// {max, sum} per workgroup.
constexpr uint32_t kEncodeRowsPerBlock = 16;      // most rows of a counting workgroup: 4 waves x 4 rows
constexpr uint32_t kEncodeFoldBlocks = 1024;      // partials a packing workgroup folds itself: 8 KB, four loads per thread
constexpr uint32_t kEncodeMaxBlocks = 65536;      // workgroups whose partials the static scratch array holds
constexpr uint32_t kEncodeHeaderBytes = 256;
constexpr uint32_t kEncodeMaxCols = (1u << 28) - 1;     // the 16 rows of a workgroup, all dense, still count in 32 bits
constexpr size_t kEncodeScratchBytes = kEncodeHeaderBytes + (size_t)kEncodeMaxBlocks * sizeof(uint2);
static_assert(kEncodeScratchBytes <= kEncodeToldOffset, "the static scratch array holds the encoder's partials");

// Rows per counting workgroup: with few rows the four waves of a workgroup share one, so that the chip is covered;
// never more partials than kEncodeFoldBlocks up to 16 384 rows.
static uint32_t encode_rows_per_block(uint32_t m) { return m <= 1024u ? 1u : m <= 4096u ? 4u : kEncodeRowsPerBlock; }

static size_t encode_scratch_bytes(uint32_t m)
{
    return kEncodeHeaderBytes + (size_t)so_ceil_div(m, encode_rows_per_block(m)) * sizeof(uint2);
}

// Four consecutive elements of a row from column j on (zeros past its end).
__device__ __forceinline__ f32x4u row_group(const float *wr, uint32_t j, uint32_t n)
{
    if (j + 4u <= n) return *reinterpret_cast<const f32x4u *>(wr + j);
    f32x4u v = {0.f, 0.f, 0.f, 0.f};
    if (j < n) v[0] = wr[j];
    if (j + 1u < n) v[1] = wr[j + 1u];
    if (j + 2u < n) v[2] = wr[j + 2u];
    return v;
}

// Pass 1: counts the entries with v != 0.0f of every row, 16 bytes per lane and eight loads in flight; the
// workgroup's maximum and sum go to partial[blockIdx.x].  Bound by the read of W: 8192 x 8192 in 43 us (6.2 TB/s;
// one word per lane and load: 188).  `sharers` = 1: a wave per row; 4: the workgroup's waves share one row.
__global__ __launch_bounds__(256)
void ellpack_count_kernel(const float *__restrict__ W, uint32_t m, uint32_t n, uint32_t *__restrict__ nnz,
                          uint2 *__restrict__ partial, uint32_t rows_per_block, uint32_t sharers)
{
    __shared__ uint32_t wmax[4], wsum[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t part = sharers == 1u ? 0u : wave;
    uint32_t vmax = 0, vsum = 0;
    for (uint32_t row = blockIdx.x * rows_per_block + (sharers == 1u ? wave : 0u); row < min(m, (blockIdx.x + 1u) * rows_per_block); row += 4u) {
        const float *wr = W + (size_t)row * n;
        uint32_t c = 0, j = part * 256u + lane * 4u;
        const uint32_t step = sharers * 256u;
        for (; j + 7u * step + 4u <= n; j += 8u * step) {
            f32x4u v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const f32x4u *>(wr + j + u * step);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) c += v[u][e] != 0.0f ? 1u : 0u;
        }
        for (; j < n; j += step) {
            const f32x4u v = row_group(wr, j, n);
#pragma unroll
            for (int e = 0; e < 4; ++e) c += v[e] != 0.0f ? 1u : 0u;
        }
        c = so_lanes::reduce<64>(c, so_lanes::Sum());
        if (sharers == 1u && lane == 0) nnz[row] = c;
        vmax = max(vmax, c);
        vsum += c;
    }
    if (lane == 0) { wmax[wave] = vmax; wsum[wave] = vsum; }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t sum = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (sharers != 1u) nnz[blockIdx.x] = sum;
        partial[blockIdx.x] = make_uint2(sharers != 1u ? sum : max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])), sum);
    }
}

// Folds the partials into header = {r, total nnz low word, high word, 0}.  One workgroup.
__global__ __launch_bounds__(1024)
void ellpack_count_fold_kernel(const uint2 *__restrict__ partial, uint32_t nblocks, uint32_t *__restrict__ header,
                               uint32_t *__restrict__ host_header)
{
    __shared__ uint32_t smax[16];
    __shared__ unsigned long long ssum[16];
    uint32_t vmax = 0;
    unsigned long long vsum = 0;
    for (uint32_t i = threadIdx.x; i < nblocks; i += 1024u) {
        const uint2 p = partial[i];
        vmax = max(vmax, p.x);
        vsum += p.y;
    }
    vmax = so_lanes::reduce<64>(vmax, so_lanes::Max());
    vsum = so_lanes::reduce<64>(vsum, so_lanes::Sum());
    if ((threadIdx.x & 63u) == 0) { smax[threadIdx.x >> 6] = vmax; ssum[threadIdx.x >> 6] = vsum; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) { vmax = max(vmax, smax[w]); vsum += ssum[w]; }
        header[0] = vmax;
        header[1] = (uint32_t)vsum;
        header[2] = (uint32_t)(vsum >> 32);
        header[3] = 0u;
        if (host_header) { host_header[0] = vmax; host_header[1] = (uint32_t)vsum; host_header[2] = (uint32_t)(vsum >> 32); }
    }
}

// Pass 2: packs (value, column) of every row in ascending column order with row pitch r, then zero-fills the
// row's remaining slots.  A lane holds four consecutive elements of each group of 256; the place of an element is
// the number of nonzeros in lower lanes (a prefix count over the wave's four ballots) plus those before it in its own
// lane.  `sharers` = 4: the workgroup's waves take a quarter each of 8192 columns at a time and tell one another their
// counts through LDS; 1: a wave per row.  Writes nothing when r exceeds r_cap (the caller's arrays hold m * r_cap
// slots); the last row's owner also clears `tail_words` words after the arrays' last slot.  Rows are taken from the
// last one back: the counting pass has left the end of W in the Infinity Cache.  `fold` != 0: r and the total come
// from that many partials (the first workgroup leaves them in the header), else from the header.
// Bound by the second read of W: 8192 x 8192, 90 % sparse, 90 -> 58 us (the whole encode, read-back included, 326 -> 127).
template <int SHARERS>
__global__ __launch_bounds__(256)
void ellpack_pack_kernel(const float *__restrict__ W, uint32_t m, uint32_t n, uint32_t *__restrict__ header, uint32_t fold,
                         uint32_t *__restrict__ host_header, uint32_t r_cap, const uint32_t *__restrict__ nnz,
                         float *__restrict__ Wd, uint32_t *__restrict__ idx, uint32_t tail_words)
{
    constexpr uint32_t G = 8;                                // groups of 256 elements a wave holds at a time
    __shared__ uint32_t smax[4], count[2][4];
    __shared__ unsigned long long ssum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t r = 0;
    if (fold == 0u) {
        r = header[0];
    } else {
        const uint2 *partial = reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(header) + kEncodeHeaderBytes);
        unsigned long long sum = 0;
        for (uint32_t i = tid; i < fold; i += 256u) { const uint2 p = partial[i]; r = max(r, p.x); sum += p.y; }
        r = so_lanes::reduce<64>(r, so_lanes::Max());
        sum = so_lanes::reduce<64>(sum, so_lanes::Sum());
        if (lane == 0) { smax[wave] = r; ssum[wave] = sum; }
        __syncthreads();
        r = max(max(smax[0], smax[1]), max(smax[2], smax[3]));
        if (blockIdx.x == 0 && tid == 0) {
            sum = ssum[0] + ssum[1] + ssum[2] + ssum[3];
            header[0] = r; header[1] = (uint32_t)sum; header[2] = (uint32_t)(sum >> 32); header[3] = 0u;
            if (host_header) { host_header[0] = r; host_header[1] = (uint32_t)sum; host_header[2] = (uint32_t)(sum >> 32); }
        }
    }
    if (r > r_cap) return;
    const uint32_t part = SHARERS == 1 ? 0u : wave;
    const uint32_t stride = SHARERS == 1 ? gridDim.x * 4u : gridDim.x;
    uint32_t turn = 0;
    for (uint32_t i = SHARERS == 1 ? blockIdx.x * 4u + wave : blockIdx.x; i < m; i += stride) {
        const uint32_t row = m - 1u - i;
        const float *wr = W + (size_t)row * n;
        float *wd = Wd + (size_t)row * r;
        uint32_t *ix = idx + (size_t)row * r;
        uint32_t base = 0;
        for (uint32_t j0 = 0; j0 < n; j0 += SHARERS * G * 256u) {
            const uint32_t jw = j0 + part * (G * 256u) + lane * 4u;
            f32x4u v[G];
            if (j0 + (part + 1u) * (G * 256u) <= n) {
#pragma unroll
                for (uint32_t u = 0; u < G; ++u) v[u] = *reinterpret_cast<const f32x4u *>(wr + jw + u * 256u);
            } else {
#pragma unroll
                for (uint32_t u = 0; u < G; ++u) v[u] = row_group(wr, jw + u * 256u, n);
            }
            if constexpr (SHARERS != 1) {
                uint32_t c = 0;
#pragma unroll
                for (uint32_t u = 0; u < G; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) c += (uint32_t)__popcll(__ballot(v[u][e] != 0.0f));
                if (lane == 0) count[turn & 1u][wave] = c;
                __syncthreads();
            }
            uint32_t at = base;
            if constexpr (SHARERS != 1) {
                const uint32_t *c = count[turn & 1u];
                const uint32_t c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
                at += wave == 0 ? 0u : wave == 1 ? c0 : wave == 2 ? c0 + c1 : c0 + c1 + c2;
                base += c0 + c1 + c2 + c3;
                ++turn;                                      // the other half of `count` next time: one barrier is enough
            }
            at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
            for (uint32_t u = 0; u < G; ++u) {
                uint64_t mask[4];
                uint32_t pos = at;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    mask[e] = __ballot(v[u][e] != 0.0f);
                    pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask[e] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask[e], pos));
                    at += (uint32_t)__popcll(mask[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v[u][e] != 0.0f) {
                        wd[pos] = v[u][e];
                        ix[pos] = jw + u * 256u + (uint32_t)e;
                        ++pos;
                    }
            }
            if constexpr (SHARERS == 1) base = at;
        }
        const uint32_t end = row + 1u == m ? r + tail_words : r;
        for (uint32_t k = nnz[row] + (SHARERS == 1 ? lane : tid); k < end; k += SHARERS * 64u) { wd[k] = 0.0f; ix[k] = 0u; }
    }
}

// The passes on the context's stream.  `scratch` holds encode_scratch_bytes(m) bytes; dWd and dIdx hold
// m * r_cap slots (+ tail_words).  `host_header` (pinned, may be null) receives r and the total once the stream has got there.
so_status encode_launch(so_ctx *ctx, const float *dDense, uint32_t m, uint32_t n, void *scratch, uint32_t r_cap,
                        uint32_t *dNnz, float *dWd, uint32_t *dIdx, uint32_t tail_words, bool count, bool pack, uint32_t *host_header)
{
    ctx->last_kernel = "encode-twice";
    uint32_t *header = (uint32_t *)scratch;
    uint2 *partial = (uint2 *)((char *)scratch + kEncodeHeaderBytes);
    const uint32_t rpb = encode_rows_per_block(m), nblocks = so_ceil_div(m, rpb);
    const bool fold_apart = !pack || m == 0 || nblocks > kEncodeFoldBlocks;
    if (count) {
        if (nblocks) {
            ellpack_count_kernel<<<nblocks, 256, 0, ctx->stream>>>(dDense, m, n, dNnz, partial, rpb, rpb == 1u ? 4u : 1u);
            SO_LAUNCH_CHECK();
        }
        if (fold_apart) {
            ellpack_count_fold_kernel<<<1, 1024, 0, ctx->stream>>>(partial, nblocks, header, host_header);
            SO_LAUNCH_CHECK();
        }
    }
    if (pack && m) {
        // A row of more than the 2048 columns that a wave holds at a time is shared by a workgroup's four waves, but where there are rows enough for all
        // waves and it is no more than twice as long.  Us, shared / a wave per row, 90 % sparse: 4072 x 1030 33.2 / 23.2, 2796 x 1500 28.4 / 21.6,
        // 2036 x 1030 24.3 / 19.2, 254 x 1030 17.7 / 17.2 (three of the four waves have nothing there); 2036 x 2060 26.1 / 22.7, 1398 x 3000 23.6 / 23.1, 1025 x 4090
        // 23.6 / 23.5, 509 x 2060 18.9 / 19.3, 254 x 2060 18.2 / 20.3.
        const uint32_t fold = count && !fold_apart ? nblocks : 0u;
        const bool shared = n > 4096u || (n > 2048u && m < 4u * (uint32_t)ctx->compute_units);
        const uint32_t blocks = std::max(1u, std::min(shared ? m : so_ceil_div(m, 4u), 16u * (uint32_t)ctx->compute_units));
        if (shared) ellpack_pack_kernel<4><<<blocks, 256, 0, ctx->stream>>>(dDense, m, n, header, fold, host_header, r_cap, dNnz, dWd, dIdx, tail_words);
        else ellpack_pack_kernel<1><<<blocks, 256, 0, ctx->stream>>>(dDense, m, n, header, fold, host_header, r_cap, dNnz, dWd, dIdx, tail_words);
        SO_LAUNCH_CHECK();
    }
    return SO_OK;
}

} // namespace

extern "C" so_status so_ellpack_encode(so_ctx *ctx, const float *dDense, uint32_t m, uint32_t n, so_ellpack **out)
{
    SO_REQUIRE(ctx && out, "so_ellpack_encode: null argument");
    *out = nullptr;
    SO_REQUIRE(dDense != nullptr || (uint64_t)m * n == 0, "so_ellpack_encode: null matrix");
    SO_REQUIRE(n <= kEncodeMaxCols, "so_ellpack_encode: at most %u columns", kEncodeMaxCols);
    so_ellpack *E = new (std::nothrow) so_ellpack();
    if (!E) { so_set_error("so_ellpack_encode: host allocation failed"); return SO_ERR_OOM; }
    E->m = m; E->n = n;
    E->layouts = SO_LAYOUT_ROW;
    void *p = nullptr, *scratch = nullptr;
    so_status s = so_malloc(ctx, (size_t)m * sizeof(uint32_t) + 16, &p);
    if (s == SO_OK) { E->d_nnz = (uint32_t *)p; s = so_fill_zero(ctx, (char *)p + (size_t)m * sizeof(uint32_t), 16); }
    if (s == SO_OK) s = so_malloc(ctx, encode_scratch_bytes(m), &scratch);
    if (s == SO_OK) s = encode_launch(ctx, dDense, m, n, scratch, 0, E->d_nnz, nullptr, nullptr, 0, true, false, ctx->h_encode_header);
    if (s == SO_OK) s = so_stream_wait(ctx, "so_ellpack_encode");
    if (s == SO_OK) {
        const uint32_t *header = ctx->h_encode_header;
        E->r = E->max_nnz = header[0];                   // r = longest row (src/ellpack_encoder.cpp:10-17)
        E->total_nnz = (uint64_t)header[1] | ((uint64_t)header[2] << 32);
        const size_t bytes = (size_t)m * E->r * sizeof(float) + 16;
        s = so_malloc(ctx, bytes, &p);
        if (s == SO_OK) { E->d_Wd = (float *)p; s = so_malloc(ctx, bytes, &p); }
        if (s == SO_OK) E->d_idx = (uint32_t *)p;
        if (s == SO_OK && (size_t)m * E->r == 0) {
            s = so_fill_zero(ctx, E->d_Wd, 16);
            if (s == SO_OK) s = so_fill_zero(ctx, E->d_idx, 16);
        }
    }
    if (s == SO_OK && (size_t)m * E->r != 0)
        s = encode_launch(ctx, dDense, m, n, scratch, E->r, E->d_nnz, E->d_Wd, E->d_idx, 4, false, true, nullptr);
    if (scratch) {
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipFree(scratch);
    }
    if (s != SO_OK) {
        (void)so_ellpack_free(ctx, E);
        return s;
    }
    *out = E;
    return SO_OK;
}

// What the kernels left in the pinned header, to the caller.
static so_status encode_counts(const so_ctx *ctx, uint32_t r_cap, uint32_t *r_out, uint64_t *total_nnz_out)
{
    const uint32_t *header = ctx->h_encode_header;
    if (r_out) *r_out = header[0];
    if (total_nnz_out) *total_nnz_out = (uint64_t)header[1] | ((uint64_t)header[2] << 32);
    SO_REQUIRE(header[0] <= r_cap, "so_ellpack_encode_noalloc: the longest row has %u nonzeros, dWd/dIdx hold %u per row (nothing was packed)",
               header[0], r_cap);
    return SO_OK;
}

extern "C" so_status so_ellpack_encode_noalloc(so_ctx *ctx, const float *dDense, uint32_t m, uint32_t n, uint32_t r_cap,
                                              float *dWd, uint32_t *dIdx, uint32_t *dNnz, uint32_t *r_out,
                                              uint64_t *total_nnz_out)
{
    SO_REQUIRE(ctx != nullptr, "so_ellpack_encode_noalloc: ctx is null");
    SO_REQUIRE(dDense != nullptr || (uint64_t)m * n == 0, "so_ellpack_encode_noalloc: null matrix");
    SO_REQUIRE(n <= kEncodeMaxCols, "so_ellpack_encode_noalloc: at most %u columns", kEncodeMaxCols);
    SO_REQUIRE(so_ceil_div(m, kEncodeRowsPerBlock) <= kEncodeMaxBlocks,
               "so_ellpack_encode_noalloc: %u rows need %u partial results, the static scratch array holds %u (at most %u rows)",
               m, so_ceil_div(m, kEncodeRowsPerBlock), kEncodeMaxBlocks, kEncodeMaxBlocks * kEncodeRowsPerBlock);
    SO_REQUIRE(m == 0 || dNnz != nullptr, "so_ellpack_encode_noalloc: dNnz is null");
    SO_REQUIRE((uint64_t)m * r_cap == 0 || (dWd != nullptr && dIdx != nullptr), "so_ellpack_encode_noalloc: dWd/dIdx is null");
    SO_REQUIRE(ctx->static_scratch != nullptr, "so_ellpack_encode_noalloc: the context has no scratch address");
    const bool counts = r_out || total_nnz_out;
    SO_REQUIRE(!counts || !ctx->capturing, "so_ellpack_encode_noalloc: r_out/total_nnz_out need a wait, which a graph recording forbids");
    // The kernels leave the counts in pinned host memory themselves: no copy to queue behind them.  A call that waits for them
    // can also be done again by the two passes if the single one says so (its workgroups wait for one another, with a bound).
    // Somebody else's kernel that made the wait reach its bound, 3 ms, is likely to be there still, or again: calls of 2^30 elements together are then
    // spared it, of twice as many each further time up to 2^34 (two passes take 0.5 to 2 us more for 2^20 elements: again some 3 ms).
    const uint64_t spared = ctx->encode_spared;
    if (counts && (uint64_t)m * r_cap != 0) {
        bool once = false;
        volatile uint32_t *at_end = nullptr;
        so_status s = so_encode_once(ctx, dDense, m, n, r_cap, dNnz, dWd, dIdx, (char *)ctx->static_scratch + kEncodeToldOffset, ctx->h_encode_header, &once, &at_end);
        if (s == SO_OK && once) s = so_tell_wait(ctx, "so_ellpack_encode_noalloc");
        if (s == SO_OK && once && *at_end != 0) s = told_wait(ctx, (uint64_t)m * n, "so_ellpack_encode_noalloc");
        if (s != SO_OK) return s;
        if (once && ctx->h_encode_header[3] == 0) {
            ctx->encode_spare_next = kEncodeSpareFirst;
            return encode_counts(ctx, r_cap, r_out, total_nnz_out);
        }
        if (once) {
            ctx->encode_spared = ctx->encode_spare_next;
            ctx->encode_spare_next = std::min(2 * ctx->encode_spare_next, kEncodeSpareMost);
        }
    }
    const so_status s = encode_launch(ctx, dDense, m, n, ctx->static_scratch, r_cap, dNnz, dWd, dIdx, 0, true,
                                      (uint64_t)m * r_cap != 0, counts ? ctx->h_encode_header : nullptr);
    if (ctx->encode_spared < spared) ctx->last_kernel = "encode-spared";
    if (s != SO_OK || !counts) return s;
    const so_status waited = told_wait(ctx, (uint64_t)m * n, "so_ellpack_encode_noalloc");
    if (waited != SO_OK) return waited;
    return encode_counts(ctx, r_cap, r_out, total_nnz_out);
}

extern "C" so_status so_ellpack_decode(so_ctx *ctx, const so_ellpack *E, float *dDense)
{
    SO_REQUIRE(ctx && E, "so_ellpack_decode: null argument");
    const size_t total = (size_t)E->m * E->n;
    if (total == 0) return SO_OK;
    SO_REQUIRE(dDense != nullptr, "so_ellpack_decode: null output");
    if (E->r == 0) return so_fill_zero(ctx, dDense, total * sizeof(float));
    const uint32_t cus = (uint32_t)ctx->compute_units;
    // Whole rows per span while they fit, but at least two spans per compute unit where the matrix has them.
    const uint32_t per_row = so_ceil_div(E->n, kDecodeSpan);
    const uint32_t rows = per_row > 1 ? 1u : std::max(1u, std::min(kDecodeSpan / E->n, so_ceil_div(E->m, 2u * cus)));
    if (rows > 1) {
        const uint32_t spans = so_ceil_div(E->m, rows);
        ellpack_decode_kernel<<<std::min(spans, 5u * cus), 256, 0, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->m, E->n, E->r, dDense, rows, spans);
    } else {
        // spans of equal width (whole cache lines), a row shared by several workgroups where there are few rows
        const uint32_t width = per_row > 1 ? so_ceil_div(so_ceil_div(E->n, per_row), 64u) * 64u : E->n, spans = so_ceil_div(E->n, width);
        const uint32_t per_seg = E->m >= 2u * cus ? spans : so_ceil_div(spans, std::min(spans, so_ceil_div(5u * cus, E->m)));
        const uint32_t segs = so_ceil_div(spans, per_seg);
        SO_REQUIRE((uint64_t)E->m * segs < (1ull << 31), "so_ellpack_decode: %u x %u is too large for one launch", E->m, E->n);
        const uint32_t items = E->m * segs, blocks = std::min(items, 5u * cus);
        if (E->ascending) ellpack_decode_wide_kernel<true><<<blocks, 256, 0, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->n, E->r, dDense, width, per_seg, segs, items);
        else ellpack_decode_wide_kernel<false><<<blocks, 256, 0, ctx->stream>>>(E->d_Wd, E->d_idx, E->d_nnz, E->n, E->r, dDense, width, per_seg, segs, items);
    }
    SO_LAUNCH_CHECK();
    return SO_OK;
}

extern "C" so_status so_ellpack_download(so_ctx *ctx, const so_ellpack *E, int layout,
                                         float *Wd, uint32_t *idx, uint32_t *nnz)
{
    SO_REQUIRE(ctx && E, "so_ellpack_download: null argument");
    SO_REQUIRE(layout == SO_LAYOUT_ROW || layout == SO_LAYOUT_SLOT,
               "so_ellpack_download: layout must be ROW or SLOT");
    SO_REQUIRE((E->layouts & layout) != 0, "so_ellpack_download: layout %d was not uploaded", layout);
    const size_t slots = (size_t)E->m * E->r;
    const float *w = layout == SO_LAYOUT_ROW ? E->d_Wd : E->d_WdT;
    const uint32_t *ix = layout == SO_LAYOUT_ROW ? E->d_idx : E->d_idxT;
    so_status s = SO_OK;
    if (Wd && slots) s = so_d2h(ctx, Wd, w, slots * sizeof(float));
    if (s == SO_OK && idx && slots) s = so_d2h(ctx, idx, ix, slots * sizeof(uint32_t));
    if (s == SO_OK && nnz && E->m) s = so_d2h(ctx, nnz, E->d_nnz, (size_t)E->m * sizeof(uint32_t));
    return s;
}
