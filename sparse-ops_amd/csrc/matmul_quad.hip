// Quad-union matmul: Y = act(E X + bias) on the matrix cores, part of layout SO_LAYOUT_RBM.
//
// Four consecutive rows (a quad) share one list of columns: the union of their nonzero columns, each
// with the four rows' weights (zero where a row has none).  v_mfma_f32_4x4x1_16b_f32 multiplies four
// weights by 64 values of an X row in 8 clocks of a SIMD, in plain fp32 with one rounding per
// multiply-add, subnormals kept (tests/test_gpu_matmul_quad.py compares with fmaf bit for bit), so one union column costs 8
// clocks per 64 dense columns whatever it holds: 2 rows' worth of useful multiply-adds at 50 % density,
// 1.58 at 30 %, 1.36 at 20 %, 1.16 at 10 %.  There is nothing to issue per nonzero -- no M0 write, no
// DPP multiply-add -- which is what bounds the row-block-merged kernel (csrc/matmul_rbm.hip).
//
// Decomposition.  A workgroup of 16 waves owns 4 * QW rows x 64 dense columns and a range of K tiles of
// 256 X rows.  A tile's 256 x 64 values are staged in LDS (64 KB, double-buffered: the next tile's loads
// are in flight while this one is multiplied); QW of the waves' worth of quads are spread over 16 / QW
// waves each, which take the quad's chunks of 16 steps in turn.  When rows x columns give too few
// workgroups the K range is split over `ks` workgroups that leave partial tiles in the context's
// workspace; the last to arrive (a counter per tile) adds them in a fixed order.
//
// One chunk = 16 steps (union columns).  A 16-byte LDS read per lane fetches four steps at once: the
// wave's quarter q (16 lanes x 4 columns = 64) reads the X row of step 4a + q, and the four MFMAs on the
// four registers read take the weights of block a of the quarter (CBSZ 2: four groups of 16 lanes, ABID
// a picks the block broadcast inside each).  Per chunk: 4 LDS reads, 16 MFMAs, one coalesced load of 64
// weights, one word of four X row bytes per quarter, four v_perm that turn them into LDS addresses.
// The quarters hold partial sums over a quarter of the steps each and are added at the end.
//
// What bounds it.  Large launches: the matrix pipe, 69 % busy at 4096 x 4096 x 256, 50 % dense (86 us;
// profiles/ellpack_matmul_quad__4096sq_c256_50pct__pmc.txt; the other 31 %: a vector instruction takes 4-5 clocks from the MFMAs, they do not overlap on a SIMD --
// 9.95 clocks per MFMA with one address add per 4 of them, 8.7 without, 8.2 with nothing but MFMAs -- and
// 0.7 us per tile of barrier, first LDS reads and the slowest wave; without the stream or the X loads the
// launch takes 87).  Small ones: latencies in a row -- launch 2.5 us, first loads 1.5, exchange of partial tiles 3.
// Two workgroups of 8 waves per compute unit with 128-row tiles instead of one of 16 measured the same or up to 5 %
// slower; the compiler's waits (it waits for all outstanding loads at every chunk) nearly twice the time.
//
// Measured, one handle launched again and again, 64 dense columns, before (row kernel) and now: 2048 x 2048 at 90 / 80 / 50 %
// sparse 9.9 / 16.9 / 35.6 us and 8.8 / 10.1 / 11.7 (0.107 GFLOP of nonzeros at 80 %: 10.7 TFLOP/s); 1024 x 1024 at 50 %
// 13.0 and 7.8; with the weights from memory 15.5 / 39.9 / 85.4 and 9.8 / 11.3 / 13.5; 25.7 and 8.1.  4096 x 784 x 256 at 90 %
// (K-tiled kernel) 15.2 and 11.9; 10 x 4096 x 256 (shared gather) 8.6 and 7.5.
//
// The order of summation differs from the reference's slot order: results agree with it to fp32
// round-off and are the same bits on every launch.  A zero weight times a non-finite X value would leave
// a NaN where the sparse product has none, so an output that comes out as NaN is computed again from the
// row's own nonzeros (`exact_outputs`): 2048 x 2048 x 64, 80 % sparse, 10.6 us, 18 with one column of NaNs in X, 125 with
// nothing else (91 and 384 with a lane per output).
#include "so_internal.h"
#include "exact_outputs.h"
#include "lds_sync.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace {

constexpr uint32_t KT = so_quads::kTileRows, WAVES = 16, LOG_WAVES = 4, TILE_BYTES = KT * 256, LDS_BYTES = 2 * TILE_BYTES + 16;
constexpr uint32_t DEPTH = 6;                     // ring slots: chunks whose weights and row bytes are requested ahead
constexpr uint32_t SLACK = so_quads::kSlack;      // chunks a wave may request past its quad's last one
static_assert((DEPTH + 2) * WAVES <= SLACK, "requests ahead stay inside the copy");

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef const u32x2 __attribute__((address_space(4))) *const_info;

struct QuadArgs {
    const float *w;             // [chunks][64]
    const uint32_t *off;        // [chunks][4]: per quarter, a byte per unit: the X row inside its tile
    const uint2 *info;          // [quads][ntiles] {first chunk, units of four steps}
    uint32_t m, n, C, nquads, ntiles;
    uint32_t qw_log2, ks, tiles_per, nslab, rbs, per_xcd;
    const float *X, *bias;
    float *Y, *part;
    uint32_t *counters;
    const float *Wd;            // the ROW arrays, for exact_outputs
    const uint32_t *idx, *nnz;
    uint32_t r;
};

// ---- the chunk loop ---------------------------------------------------------------------------------
//
// A wave's chunks of one tile, as one block of assembly, because its waits need counting by hand: the
// weights and X row bytes of a chunk are requested DEPTH chunks ahead (they come from memory once, so
// memory's latency has to be covered, not L2's) into a ring of registers, across tile boundaries, and the
// compiler's own waits would assume the worst over all ways into a ring slot, which is to wait for everything.
// The ring (v84 .. v95) is also in flight between the blocks, where the compiler believes its registers hold values: it
// must neither move nor spill them there, nor issue vector memory instructions of its own, which the waits would count.
// csrc/check_quad_ring.py looks for both in the assembly of every build.
//
//   ENTER_S  the run starts at ring slot S: LDS reads of its chunk
//   CHUNK_S  `n` chunks left, this one's LDS reads under way.  Slot S+1's requests have at least
//            2 * (DEPTH - 2) younger ones; the next chunk's reads go out, then this chunk's 16 MFMAs.
//   LAST_S   the run's last chunk: only its first `last` units hold steps
//
// LDS returns data in order, so lgkmcnt(7 .. 4) waits for this chunk's reads and leaves the next one's in
// flight.  An accumulator comes up every fourth MFMA.
#define SO_MF(W, X, A, U) "v_mfma_f32_4x4x1_16b_f32 " A ", " W ", " X ", " A " cbsz:2 abid:" U "\n\t"
#define SO_UNIT(W, X0, X1, X2, X3, U) SO_MF(W, X0, "v[32:35]", U) SO_MF(W, X1, "v[36:39]", U) SO_MF(W, X2, "v[40:43]", U) SO_MF(W, X3, "v[44:47]", U)
// the LDS operands of a chunk: v48 .. v63 for even ring slots, v64 .. v79 for odd ones
#define SO_UNITS_A0(W) SO_UNIT(W, "v48", "v49", "v50", "v51", "0")
#define SO_UNITS_A1(W) SO_UNIT(W, "v52", "v53", "v54", "v55", "1")
#define SO_UNITS_A2(W) SO_UNIT(W, "v56", "v57", "v58", "v59", "2")
#define SO_UNITS_A3(W) SO_UNIT(W, "v60", "v61", "v62", "v63", "3")
#define SO_UNITS_B0(W) SO_UNIT(W, "v64", "v65", "v66", "v67", "0")
#define SO_UNITS_B1(W) SO_UNIT(W, "v68", "v69", "v70", "v71", "1")
#define SO_UNITS_B2(W) SO_UNIT(W, "v72", "v73", "v74", "v75", "2")
#define SO_UNITS_B3(W) SO_UNIT(W, "v76", "v77", "v78", "v79", "3")
#define SO_READ_A "ds_read_b128 v[48:51], v80\n\tds_read_b128 v[52:55], v81\n\tds_read_b128 v[56:59], v82\n\tds_read_b128 v[60:63], v83\n\t"
#define SO_READ_B "ds_read_b128 v[64:67], v80\n\tds_read_b128 v[68:71], v81\n\tds_read_b128 v[72:75], v82\n\tds_read_b128 v[76:79], v83\n\t"
// LDS addresses of the four units' X rows: byte 0 the lane's place in the row, byte 1 the row, byte 2 the buffer
#define SO_ADDR(O) "v_perm_b32 v80, " O ", %[base], %[s0]\n\tv_perm_b32 v81, " O ", %[base], %[s1]\n\t" \
                   "v_perm_b32 v82, " O ", %[base], %[s2]\n\tv_perm_b32 v83, " O ", %[base], %[s3]\n\t"
#define SO_ASK(W, O) "global_load_dword " W ", %[lane4], s[40:41]\n\tglobal_load_dword " O ", %[quarter4], s[42:43]\n\t" \
                     "s_add_u32 s40, s40, %[wstep]\n\ts_addc_u32 s41, s41, 0\n\ts_add_u32 s42, s42, %[ostep]\n\ts_addc_u32 s43, s43, 0\n\t"
#define SO_ENTER(S, X, O) "Lenter" S "_%=:\n\ts_waitcnt vmcnt(10)\n\t" SO_ADDR(O) SO_READ_##X "s_branch Lchunk" S "_%=\n\t"
#define SO_CHUNK(S, N, X, Y, W, O, ON)                                                                       \
    "Lchunk" S "_%=:\n\ts_sub_u32 %[n], %[n], 1\n\t"                                                          \
    "s_cmp_eq_u32 %[n], 0\n\ts_cbranch_scc1 Llast" S "_%=\n\ts_waitcnt vmcnt(8)\n\t"                       \
    SO_ADDR(ON) SO_READ_##Y                                                                                  \
    "s_waitcnt lgkmcnt(7)\n\t" SO_UNITS_##X##0(W) "s_waitcnt lgkmcnt(6)\n\t" SO_UNITS_##X##1(W)              \
    "s_waitcnt lgkmcnt(5)\n\t" SO_UNITS_##X##2(W) "s_waitcnt lgkmcnt(4)\n\t" SO_UNITS_##X##3(W)              \
    SO_ASK(W, O)
#define SO_LAST(S, N, X, W, O)                                                                               \
    "Llast" S "_%=:\n\ts_mov_b32 %[phase], " N "\n\ts_waitcnt lgkmcnt(0)\n\t" SO_UNITS_##X##0(W)             \
    "s_cmp_lt_u32 %[last], 2\n\ts_cbranch_scc1 Lask" S "_%=\n\t" SO_UNITS_##X##1(W)                         \
    "s_cmp_lt_u32 %[last], 3\n\ts_cbranch_scc1 Lask" S "_%=\n\t" SO_UNITS_##X##2(W)                         \
    "s_cmp_lt_u32 %[last], 4\n\ts_cbranch_scc1 Lask" S "_%=\n\t" SO_UNITS_##X##3(W)                         \
    "Lask" S "_%=:\n\t" SO_ASK(W, O) "s_branch Lend_%=\n\t"
#define SO_QUAD_LOOP                                                                                         \
    "s_cmp_eq_u32 %[phase], 0\n\ts_cbranch_scc1 Lenter0_%=\n\ts_cmp_eq_u32 %[phase], 1\n\ts_cbranch_scc1 Lenter1_%=\n\t" \
    "s_cmp_eq_u32 %[phase], 2\n\ts_cbranch_scc1 Lenter2_%=\n\ts_cmp_eq_u32 %[phase], 3\n\ts_cbranch_scc1 Lenter3_%=\n\t" \
    "s_cmp_eq_u32 %[phase], 4\n\ts_cbranch_scc1 Lenter4_%=\n\ts_branch Lenter5_%=\n\t"                     \
    SO_ENTER("0", A, "v90") SO_ENTER("1", B, "v91") SO_ENTER("2", A, "v92")                                  \
    SO_ENTER("3", B, "v93") SO_ENTER("4", A, "v94") SO_ENTER("5", B, "v95")                                  \
    SO_CHUNK("0", "1", A, B, "v84", "v90", "v91") SO_CHUNK("1", "2", B, A, "v85", "v91", "v92")              \
    SO_CHUNK("2", "3", A, B, "v86", "v92", "v93") SO_CHUNK("3", "4", B, A, "v87", "v93", "v94")              \
    SO_CHUNK("4", "5", A, B, "v88", "v94", "v95") SO_CHUNK("5", "0", B, A, "v89", "v95", "v90")              \
    "s_branch Lchunk0_%=\n\t"                                                                               \
    SO_LAST("0", "1", A, "v84", "v90") SO_LAST("1", "2", B, "v85", "v91") SO_LAST("2", "3", A, "v86", "v92") \
    SO_LAST("3", "4", B, "v87", "v93") SO_LAST("4", "5", A, "v88", "v94") SO_LAST("5", "0", B, "v89", "v95") \
    "Lend_%=:\n\ts_nop 7"      /* the accumulators may be read by vector instructions from here on */

template <int ACT>
__global__ __launch_bounds__(WAVES * 64)
void ellpack_matmul_quad_kernel(QuadArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, quarter = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup ids go round the 8 XCDs; an XCD takes a contiguous share of the (row block, K part, slab)
    // triples, so the workgroups that walk the same weights, and those that exchange partial tiles, share an L2.
    const uint32_t combos = a.nslab * a.ks, id = (blockIdx.x & 7u) * a.per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= a.per_xcd || id >= a.rbs * combos) return;
    const uint32_t rb = id / combos, combo = id - rb * combos;
    const uint32_t kp = combo / a.nslab, slab = combo - kp * a.nslab;
    const uint32_t qw = 1u << a.qw_log2, kw = WAVES >> a.qw_log2;
    const uint32_t wq = wave & (qw - 1u), wk = wave >> a.qw_log2;
    const uint32_t quad = (rb << a.qw_log2) + wq;                   // the waves of one quad: wq + i * qw
    const bool has_quad = quad < a.nquads;
    const uint32_t t0 = kp * a.tiles_per, t1 = min(a.ntiles, t0 + a.tiles_per);

    // X staging, straight from memory into LDS: 16 lanes x 16 bytes per row, four rows per wave and load, 64 rows
    // per round of the workgroup.  Groups of four columns past the last column repeat the slab's first group and
    // rows past the last row repeat it (neither is ever used); a group that would end past the end of X (C not a
    // multiple of 4, last row) is read from where four values are left and shifted once it is in LDS.
    const uint32_t sgrp = (tid & 15u) * 4u, srow = tid >> 4, pitch = a.C;
    const uint32_t xgrp = slab * 64u + (slab * 64u + sgrp < a.C ? sgrp : 0u);
    const bool overhang = a.C % 4u != 0u && slab + 1u == a.nslab;
    const uint32_t lds0 = so_lds::lds_address(lds);
    auto place = [&](uint32_t t, uint32_t k) { return min(k * 64u + srow, a.n - 1u - t * KT) * pitch + xgrp; };   // element of X from the tile's first row on
    auto ends = [&](uint32_t t) { return (uint32_t)min((uint64_t)(a.n - t * KT) * pitch - 4u, (uint64_t)0x3ffffff0u); };   // the last place four values can be read from
    // byte offsets of this thread's four loads from the tile's first X row on; only in the last tile, where rows or
    // values may run out, do they differ
    uint32_t at0 = (srow * pitch + xgrp) * 4u, at1 = at0 + 256u * pitch, at2 = at1 + 256u * pitch, at3 = at2 + 256u * pitch;
    auto fetch = [&](uint32_t t) {
        const float *p = a.X + (size_t)t * KT * pitch;
        const uint32_t to = lds0 + ((t - t0) & 1u) * TILE_BYTES + wave * 1024u;
        if (t + 2u >= a.ntiles) {                 // the last tile, or one whose last groups could reach past it
            const uint32_t e = ends(t);
            at0 = min(place(t, 0), e) * 4u; at1 = min(place(t, 1), e) * 4u; at2 = min(place(t, 2), e) * 4u; at3 = min(place(t, 3), e) * 4u;
        }
        asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %4\n\ts_add_u32 m0, %5, 0x4000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %4\n\t"
                     "s_add_u32 m0, %5, 0x8000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4\n\ts_add_u32 m0, %5, 0xc000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %4"
                     : : "v"(at0), "v"(at1), "v"(at2), "v"(at3), "s"(p), "s"(to) : "memory", "m0", "scc");
    };
    // Waits for this wave's part of tile t; `younger` = chunks requested since, two loads each.
    auto fetched = [&](uint32_t t, uint32_t younger) {
        if (younger >= 4u) asm volatile("s_waitcnt vmcnt(8)" : : : "memory");
        else if (younger >= 2u) asm volatile("s_waitcnt vmcnt(4)" : : : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        if (overhang && t + 1u == a.ntiles) {
            const uint32_t e = ends(t);
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t at = place(t, k);
                if (at > e) {
                    f32x4 *p = reinterpret_cast<f32x4 *>(lds + ((t - t0) & 1u) * TILE_BYTES + (k * 1024u + tid) * 16u);
                    const f32x4 u = *p;
                    const uint32_t shift = at - e;
                    *p = f32x4{shift == 1u ? u[1] : shift == 2u ? u[2] : u[3], shift == 1u ? u[2] : u[3], u[3], u[3]};
                }
            }
        }
    };

    f32x4 acc[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};

    fetch(t0);
    // (through the constant address space: scalar loads also next to inline assembly)
    const const_info inf = (const_info)(uintptr_t)(a.info + (size_t)(has_quad ? quad : 0u) * a.ntiles);
    u32x2 cur = inf[t0], next = inf[min(t0 + 1u, a.ntiles - 1u)];
    uint32_t c = cur.x + ((wk - (cur.x - inf[0].x)) & (kw - 1u));     // the wave's next chunk: every kw-th of the quad's is its turn
    const float *wp = a.w + (size_t)c * 64u;
    const uint32_t *op = a.off + (size_t)c * 4u;
    const uint32_t wstep = 256u * kw, ostep = 16u * kw, lane4 = lane * 4u, quarter4 = quarter * 4u;
    float w0, w1, w2, w3, w4, w5;
    uint32_t o0, o1, o2, o3, o4, o5;
    asm volatile("; ring: first requests\n\t" SO_ASK("v84", "v90") SO_ASK("v85", "v91") SO_ASK("v86", "v92") SO_ASK("v87", "v93") SO_ASK("v88", "v94") SO_ASK("v89", "v95")
                 : "={v84}"(w0), "={v85}"(w1), "={v86}"(w2), "={v87}"(w3), "={v88}"(w4), "={v89}"(w5), "={v90}"(o0), "={v91}"(o1), "={v92}"(o2),
                   "={v93}"(o3), "={v94}"(o4), "={v95}"(o5), "+{s[40:41]}"(wp), "+{s[42:43]}"(op)
                 : [lane4] "v"(lane4), [quarter4] "v"(quarter4), [wstep] "s"(wstep), [ostep] "s"(ostep) : "memory", "scc");
    fetched(t0, DEPTH);
    __syncthreads();
    if (t0 + 1u < t1) fetch(t0 + 1u);

    uint32_t phase = 0;
    for (uint32_t t = t0;;) {
        const uint32_t base = so_lds::lds_address(lds) + (lane & 15u) * 16u + (((t - t0) & 1u) << 16);
        const uint32_t end = cur.x + ((cur.y + 3u) >> 2);
        uint32_t n = has_quad && c < end ? (end - c + kw - 1u) >> (LOG_WAVES - a.qw_log2) : 0u;
        const uint32_t taken = n;
        if (n != 0u) {
            c += n * kw;
            const uint32_t last = c - kw + 1u == end ? cur.y - 4u * (end - 1u - cur.x) : 4u;    // units in the wave's last chunk
            asm volatile(SO_QUAD_LOOP
                         : "+{v[32:35]}"(acc[0]), "+{v[36:39]}"(acc[1]), "+{v[40:43]}"(acc[2]), "+{v[44:47]}"(acc[3]),
                           "+{v84}"(w0), "+{v85}"(w1), "+{v86}"(w2), "+{v87}"(w3), "+{v88}"(w4), "+{v89}"(w5),
                           "+{v90}"(o0), "+{v91}"(o1), "+{v92}"(o2), "+{v93}"(o3), "+{v94}"(o4), "+{v95}"(o5),
                           "+{s[40:41]}"(wp), "+{s[42:43]}"(op), [n] "+s"(n), [phase] "+s"(phase)
                         : [lane4] "v"(lane4), [quarter4] "v"(quarter4), [base] "v"(base), [wstep] "s"(wstep), [ostep] "s"(ostep), [last] "s"(last),
                           [s0] "s"(0x0c020400u), [s1] "s"(0x0c020500u), [s2] "s"(0x0c020600u), [s3] "s"(0x0c020700u)
                         : "memory", "scc", "v48", "v49", "v50", "v51", "v52", "v53", "v54", "v55", "v56", "v57", "v58", "v59", "v60", "v61", "v62", "v63",
                           "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79",
                           "v80", "v81", "v82", "v83");
        }
        if (++t >= t1) break;
        cur = next;
        next = inf[min(t + 1u, a.ntiles - 1u)];
        fetched(t, taken);
        __syncthreads();
        if (t + 1u < t1) fetch(t + 1u);
    }
    // the ring's last requests (and a tail fetch, none): nothing is outstanding from here on
    asm volatile("; ring: drained\n\ts_waitcnt vmcnt(0)" : "+{v84}"(w0), "+{v85}"(w1), "+{v86}"(w2), "+{v87}"(w3), "+{v88}"(w4), "+{v89}"(w5), "+{v90}"(o0), "+{v91}"(o1),
                 "+{v92}"(o2), "+{v93}"(o3), "+{v94}"(o4), "+{v95}"(o5) : : "memory");

    // Sum over the quarters: after the two exchanges quarter q of the wave holds row q, four columns per lane.
    f32x4 s;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const u32x2 p = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[v][0]), __float_as_uint(acc[v][2]), false, false);
        const u32x2 q = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[v][1]), __float_as_uint(acc[v][3]), false, false);
        const float s02 = __uint_as_float(p[0]) + __uint_as_float(p[1]), s13 = __uint_as_float(q[0]) + __uint_as_float(q[1]);
        const u32x2 e = __builtin_amdgcn_permlane16_swap(__float_as_uint(s02), __float_as_uint(s13), false, false);
        s[v] = __uint_as_float(e[0]) + __uint_as_float(e[1]);
    }
    // Sum over the waves of a quad, through LDS.
    if (kw > 1u) {
        f32x4 *red = reinterpret_cast<f32x4 *>(lds);
        __syncthreads();
        red[wave * 64u + lane] = s;
        __syncthreads();
        if (wk == 0) for (uint32_t k = 1; k < kw; ++k) s += red[((k << a.qw_log2) + wq) * 64u + lane];
    }
    const uint32_t tile = rb * a.nslab + slab;
    if (a.ks > 1u) {
        f32x4 *mine = reinterpret_cast<f32x4 *>(a.part) + ((size_t)tile * a.ks + kp) * (qw * 64u) + wq * 64u + lane;
        // sc1: written through to memory, whichever XCD the tile's other workgroups run on
        if (wk == 0) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : : "v"(mine), "v"(s) : "memory");
        __syncthreads();
        uint32_t *arrived = reinterpret_cast<uint32_t *>(lds + 2 * TILE_BYTES);
        if (tid == 0) *arrived = __hip_atomic_fetch_add(&a.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*arrived != a.ks - 1u) return;                     // the last workgroup of the tile to arrive finishes it
        if (tid == 0) __hip_atomic_store(&a.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
        // wave wk of a quad adds the parts wk, wk + kw, ...; then the waves' sums are added as above
        s = f32x4{0.f, 0.f, 0.f, 0.f};
        const f32x4 *p = reinterpret_cast<const f32x4 *>(a.part) + (size_t)tile * a.ks * (qw * 64u) + wq * 64u + lane;
        for (uint32_t k = wk; k < a.ks; k += 4u * kw) {
            f32x4 v[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (k + i * kw < a.ks) asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v[i]) : "v"(p + (size_t)(k + i * kw) * (qw * 64u)) : "memory");
            }
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : : "memory");
            s += v[0]; s += v[1]; s += v[2]; s += v[3];
        }
        if (kw > 1u) {
            f32x4 *red = reinterpret_cast<f32x4 *>(lds);
            red[wave * 64u + lane] = s;
            __syncthreads();
            if (wk == 0) for (uint32_t k = 1; k < kw; ++k) s += red[((k << a.qw_log2) + wq) * 64u + lane];
        }
    }
    if (wk != 0 || !has_quad) return;
    const uint32_t sub = lane & 15u, row = quad * 4u + quarter, col = slab * 64u + sub * 4u;
    // outputs that came out as NaN, a group of four columns (of all four rows) at a time
    const bool lost = row < a.m && ((__builtin_isnan(s[0]) && col < a.C) || (__builtin_isnan(s[1]) && col + 1u < a.C) ||
                                    (__builtin_isnan(s[2]) && col + 2u < a.C) || (__builtin_isnan(s[3]) && col + 3u < a.C));
    uint64_t groups = __ballot(lost);
    groups |= groups >> 32;
    for (uint32_t left = (uint32_t)(groups | groups >> 16) & 0xffffu; left != 0u; left &= left - 1u) {
        const uint32_t g = (uint32_t)__builtin_ctz(left);
        const uint32_t first = min(slab * 64u + g * 4u, a.C - 4u), past = slab * 64u + g * 4u - first;   // four columns that exist
        f32x4 e = exact_outputs(a, row, first, sub);
        if (past != 0u) e = f32x4{past == 1u ? e[1] : past == 2u ? e[2] : e[3], past == 1u ? e[2] : e[3], e[3], e[3]};
#pragma unroll
        for (int v = 0; v < 4; ++v) s[v] = g == sub && __builtin_isnan(s[v]) ? e[v] : s[v];
    }
    if (row >= a.m || col >= a.C) return;
    const float b = a.bias ? a.bias[row] : 0.0f;
    f32x4 y;
#pragma unroll
    for (int v = 0; v < 4; ++v) y[v] = so_epilogue<ACT>(s[v] + b);
    float *yp = a.Y + (size_t)row * a.C + col;
    if (col + 4u <= a.C) *reinterpret_cast<f32x4u *>(yp) = y;
    else {
        yp[0] = y[0];
        if (col + 1u < a.C) yp[1] = y[1];
        if (col + 2u < a.C) yp[2] = y[2];
    }
}

} // namespace

// Rows per workgroup and K split by estimated time (us).  The model -- rounds of one workgroup per compute unit,
// each with its start-up and, per tile, the larger of the multiply-adds and of what a tile's X values take to
// arrive; for a split the exchange of partial tiles -- was fitted to launches of 10..4096 rows, 512..4096 columns, 4..256
// dense columns, 50-95 % sparse.  Over the 18 shapes of profiles/matmul_quad__plans.txt its choice takes 1.4 % longer than the
// best of all plans on average, 6 % at most.
so_quad_plan so_matmul_quad_choose(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    const so_quads &Q = E->quads;
    so_quad_plan best{};
    best.us = 1e30;
    const uint32_t nslab = so_ceil_div(C, 64);
    const double units = (double)Q.total_units / ((double)Q.nquads * Q.ntiles), cus = ctx->compute_units;
    for (uint32_t ql = 0; ql <= LOG_WAVES; ++ql) {
        const uint32_t rbs = so_ceil_div(Q.nquads, 1u << ql);
        for (uint32_t ks = 1; ks <= Q.ntiles && ks <= so_quads::kMaxSplit; ks += ks < 4 ? 1 : ks / 2) {
            const uint32_t tiles_per = so_ceil_div(Q.ntiles, ks), parts = so_ceil_div(Q.ntiles, tiles_per);
            const double wgs = (double)rbs * nslab * parts;
            const double full = std::min(1.0, wgs / cus), sustained = std::min(1.0, tiles_per / 8.0);   // long launches on the whole chip run at lower clocks
            const double multiply = 0.68 + (0.0635 + 0.01 * full * sustained) / WAVES * units * (1u << ql);
            const double tile = std::max(multiply, 0.42 * (0.4 + 0.6 * full));
            // (kQuadLeastUs: one round, one tile)
            const double us = std::ceil(wgs / cus) * (3.8 + tiles_per * tile) + (parts > 1 ? 1.75 + 0.007 * (1u << ql) * parts : 0.0);
            if (us < best.us) best = so_quad_plan{ql, parts, tiles_per, nslab, rbs, us};
        }
    }
    if (ctx->tune.matmul_quad_rows >= 0 && ctx->tune.matmul_quad_rows <= (int)LOG_WAVES) {
        best.qw_log2 = (uint32_t)ctx->tune.matmul_quad_rows;
        best.rbs = so_ceil_div(Q.nquads, 1u << best.qw_log2);
    }
    if (ctx->tune.matmul_quad_split > 0) {
        best.tiles_per = so_ceil_div(Q.ntiles, std::min<uint32_t>(std::min(Q.ntiles, so_quads::kMaxSplit), (uint32_t)ctx->tune.matmul_quad_split));
        best.ks = so_ceil_div(Q.ntiles, best.tiles_per);
    }
    return best;
}

namespace {

template <int ACT>
so_status launch_quad(so_ctx *ctx, const QuadArgs &a, uint32_t blocks)
{
    SO_HIP(so_allow_big_lds(ctx, (const void *)ellpack_matmul_quad_kernel<ACT>));
    ellpack_matmul_quad_kernel<ACT><<<blocks, WAVES * 64, LDS_BYTES, ctx->stream>>>(a);
    return SO_OK;
}

size_t part_bytes(const so_quad_plan &p) { return (size_t)p.rbs * p.nslab * p.ks * (1u << p.qw_log2) * 64 * 16; }
size_t counter_bytes(const so_quad_plan &p) { return (size_t)p.rbs * p.nslab * sizeof(uint32_t); }

so_status workspace(so_ctx *ctx, const so_ellpack *E, uint32_t C, const so_quad_plan &p)
{
    if (p.ks == 1) return SO_OK;
    SO_REQUIRE((uint64_t)p.rbs * p.nslab * p.ks < (1ull << 28), "so_matmul: %u x %u output is too large for one launch", E->m, C);
    return so_matmul_workspace(ctx, part_bytes(p), counter_bytes(p));
}

// ------------------------------------------------------------------ the builder

struct Entry { uint32_t col, row; float w; };

// rows: the X row of every step, from its tile and its byte there; zeros for the slack.  16 lanes per (quad, tile) run.  (Made here: written and
// copied by the host with the rest, they took a tenth of an upload's time.)
__global__ __launch_bounds__(256)
void quad_rows_kernel(uint16_t *rows, uint64_t chunks, const uint8_t *off, const uint2 *info, uint64_t runs, uint32_t ntiles)
{
    const uint32_t sub = threadIdx.x & 15u;
    for (uint64_t i = blockIdx.x * 16ull + (threadIdx.x >> 4); i <= runs; i += gridDim.x * 16ull) {
        const uint2 run = info[i < runs ? i : runs - 1u];
        const uint64_t past = run.x + (uint64_t)((run.y + 3u) >> 2);
        if (i < runs) for (uint64_t c = run.x; c < past; ++c) rows[c * 16u + sub] = (uint16_t)(i % ntiles * KT + off[c * 16u + sub]);
        else for (uint64_t c = past; c < chunks; ++c) rows[c * 16u + sub] = 0u;
    }
}

// Rows with ascending columns: tile(t, mask, weights) for every tile of quad q, with a bit per union column and, where
// WEIGHTS, the four weights of each (weights[4 * column ..], zeros elsewhere: tile puts back zeros where it takes them).
template <bool WEIGHTS, class F>
void walk_tiles(const so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz, uint32_t q, float *weights, F &&tile)
{
    static_assert(KT == 256, "four words of columns per tile");
    const uint32_t r0 = q * 4, rows = std::min(4u, E->m - r0);
    uint32_t pos[4] = {0, 0, 0, 0};
    for (uint32_t t = 0; t < E->quads.ntiles; ++t) {
        const uint32_t base = t * KT;
        uint64_t mask[4] = {0, 0, 0, 0};
        for (uint32_t i = 0; i < rows; ++i) {
            const uint32_t *ix = idx + (size_t)(r0 + i) * E->r;
            const float *wd = Wd + (size_t)(r0 + i) * E->r;
            uint32_t k = pos[i];
            for (; k < nnz[r0 + i] && ix[k] - base < KT; ++k) {
                const uint32_t c = ix[k] - base;
                mask[c >> 6] |= 1ull << (c & 63);
                if (WEIGHTS) weights[4 * c + i] = wd[k];
            }
            pos[i] = k;
        }
        tile(t, mask, weights);
    }
}

// Rows in any order: the union columns of quad q, ascending, with up to four weights each (a column that a row names
// twice gets two steps): calls step(col, weights) for every step.
template <class F>
void walk_quad(const so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz, uint32_t q, std::vector<Entry> &tmp, F &&step)
{
    const uint32_t r0 = q * 4, rows = std::min(4u, E->m - r0);
    tmp.clear();
    for (uint32_t i = 0; i < rows; ++i)
        for (uint32_t k = 0; k < nnz[r0 + i]; ++k) tmp.push_back({idx[(size_t)(r0 + i) * E->r + k], i, Wd[(size_t)(r0 + i) * E->r + k]});
    std::stable_sort(tmp.begin(), tmp.end(), [](const Entry &a, const Entry &b) { return a.col < b.col; });
    for (size_t k = 0; k < tmp.size();) {
        float w[4] = {0.f, 0.f, 0.f, 0.f};
        uint32_t have = 0;
        const uint32_t col = tmp[k].col;
        for (; k < tmp.size() && tmp[k].col == col && !(have & (1u << tmp[k].row)); ++k) { w[tmp[k].row] = tmp[k].w; have |= 1u << tmp[k].row; }
        step(col, w);
    }
}

} // namespace

so_status so_quads_build(so_ctx *ctx, so_ellpack *E, const float *Wd, const uint32_t *idx, const uint32_t *nnz)
{
    so_quads &Q = E->quads;
    Q.nquads = so_ceil_div(E->m, 4);
    Q.ntiles = std::max(1u, so_ceil_div(E->n, KT));
    // The tables have an entry per (quad, tile) and a run of columns there is at least one chunk of 272 bytes, so the copy
    // of a very sparse matrix is many times the matrix (65536 x 65536, 10 nonzeros a row: 270 MB beside 5), while the
    // kernel would multiply padding: such a handle does without.  Four times the nonzeros' values and columns is
    // reached at about 8 nonzeros per run (99.2 % sparse); a mebibyte is no matter.
    const uint64_t most = std::max<uint64_t>(1u << 20, 32 * E->total_nnz);
    if ((uint64_t)Q.nquads * Q.ntiles * sizeof(uint2) > most) { Q = so_quads(); return SO_OK; }
    std::vector<uint32_t> steps((size_t)Q.nquads * Q.ntiles, 0);
    so_parallel(Q.nquads, E->total_nnz, [&](uint32_t q0, uint32_t q1) {
        std::vector<Entry> tmp;
        for (uint32_t q = q0; q < q1; ++q) {
            uint32_t *const count = steps.data() + (size_t)q * Q.ntiles;
            if (E->ascending)
                walk_tiles<false>(E, Wd, idx, nnz, q, nullptr, [&](uint32_t t, const uint64_t *mask, float *) {
                    for (int k = 0; k < 4; ++k) count[t] += (uint32_t)__builtin_popcountll(mask[k]);
                });
            else walk_quad(E, Wd, idx, nnz, q, tmp, [&](uint32_t col, const float *) { ++count[col / KT]; });
        }
    });
    std::vector<uint2> info(steps.size());
    uint64_t chunks = 0;
    Q.total_units = 0;
    for (size_t k = 0; k < steps.size(); ++k) {
        const uint32_t units = (steps[k] + 3) / 4;
        info[k] = make_uint2((uint32_t)chunks, units);
        chunks += (units + 3) / 4;
        Q.total_units += units;
    }
    Q.total_chunks = chunks;
    if (chunks > 0xfffff000ull || chunks * 272 + info.size() * sizeof(uint2) > most) { Q = so_quads(); return SO_OK; }
    // padding steps: zero weights on the tile's first row
    // (the three arrays in one allocation and one copy: each of either costs a small matrix a tenth of a millisecond)
    const size_t w_bytes = (size_t)(chunks + SLACK) * 256, off_bytes = (size_t)(chunks + SLACK) * 16;
    std::vector<uint8_t> blob(w_bytes + off_bytes + info.size() * sizeof(uint2), 0u);
    float *w = reinterpret_cast<float *>(blob.data());
    uint8_t *off = blob.data() + w_bytes;
    std::memcpy(off + off_bytes, info.data(), info.size() * sizeof(uint2));
    so_parallel(Q.nquads, E->total_nnz, [&](uint32_t q0, uint32_t q1) {
        std::vector<Entry> tmp;
        std::vector<float> weights(4 * KT, 0.0f);
        const auto put = [&](size_t s, uint32_t c, const float *wt) {       // step s: column c of its tile
            const size_t chunk = s >> 4, unit = (s >> 2) & 3, quarter = s & 3;
            std::memcpy(w + chunk * 64 + quarter * 16 + unit * 4, wt, 16);
            off[chunk * 16 + quarter * 4 + unit] = (uint8_t)c;
        };
        for (uint32_t q = q0; q < q1; ++q) {
            const uint2 *const runs = info.data() + (size_t)q * Q.ntiles;
            uint32_t tile = 0xffffffffu;
            size_t s = 0;
            if (E->ascending)
                walk_tiles<true>(E, Wd, idx, nnz, q, weights.data(), [&](uint32_t t, const uint64_t *mask, float *wt) {
                    s = (size_t)runs[t].x * 16;
                    for (uint32_t k = 0; k < 4; ++k)
                        for (uint64_t left = mask[k]; left != 0; left &= left - 1) {
                            const uint32_t c = k * 64 + (uint32_t)__builtin_ctzll(left);
                            put(s++, c, wt + 4 * c);
                            std::memset(wt + 4 * c, 0, 16);
                        }
                });
            else
                walk_quad(E, Wd, idx, nnz, q, tmp, [&](uint32_t col, const float *wt) {
                    if (col / KT != tile) { tile = col / KT; s = (size_t)runs[tile].x * 16; }
                    put(s++, col - tile * KT, wt);
                });
        }
    });
    void *p = nullptr;
    const size_t rows_bytes = E->n <= so_quads::kMostRows ? 2 * off_bytes : 0, rows_at = (blob.size() + 15) & ~(size_t)15;
    so_status s = so_malloc(ctx, rows_at + rows_bytes, &p);
    if (s != SO_OK) { Q = so_quads(); return s; }
    Q.d_w = (float *)p;
    Q.d_off = (uint32_t *)((char *)p + w_bytes);
    Q.d_info = (uint2 *)((char *)p + w_bytes + off_bytes);
    s = so_h2d(ctx, p, blob.data(), blob.size());
    if (s != SO_OK || rows_bytes == 0 || info.empty()) return s;
    Q.d_rows = (uint16_t *)((char *)p + rows_at);
    const uint64_t runs = (uint64_t)Q.nquads * Q.ntiles;
    quad_rows_kernel<<<(uint32_t)std::min<uint64_t>((runs + 16) / 16, 65536), 256, 0, ctx->stream>>>(Q.d_rows, off_bytes / 16, (const uint8_t *)Q.d_off, Q.d_info, runs, Q.ntiles);
    SO_LAUNCH_CHECK();
    return so_stream_wait(ctx, "so_ellpack_upload");
}

void so_quads_free(so_ellpack *E)
{
    so_quads &Q = E->quads;
    if (Q.d_w) (void)hipFree(Q.d_w);
    Q = so_quads();
}

bool so_matmul_quad_applies(const so_ctx *ctx, const so_ellpack *E, uint32_t C)
{
    return E->quads.d_w != nullptr && E->n != 0 && C >= 4 && C < (1u << 21) && (size_t)ctx->max_lds_bytes >= LDS_BYTES;
}

so_status so_matmul_quad_reserve(so_ctx *ctx, const so_ellpack *E, uint32_t C) { return workspace(ctx, E, C, so_matmul_quad_choose(ctx, E, C)); }

bool so_matmul_quad_ready(const so_ctx *ctx, const so_quad_plan &p)
{
    return p.ks == 1 || (ctx->mm_part && ctx->mm_counters && part_bytes(p) <= ctx->mm_part->bytes && counter_bytes(p) <= ctx->mm_counters->bytes);
}

so_status so_matmul_quad_launch(so_ctx *ctx, const so_ellpack *E, const so_quad_plan &p, const float *dX, uint32_t C, const float *dBias, float *dY, int act)
{
    const so_status s = workspace(ctx, E, C, p);
    if (s != SO_OK) return s;
    const so_quads &Q = E->quads;
    const uint32_t per_xcd = so_ceil_div((uint64_t)p.rbs * p.nslab * p.ks, 8);
    const QuadArgs a{Q.d_w, Q.d_off, Q.d_info, E->m, E->n, C, Q.nquads, Q.ntiles, p.qw_log2, p.ks, p.tiles_per, p.nslab, p.rbs, per_xcd,
                     dX, dBias, dY, ctx->mm_part ? (float *)ctx->mm_part->p : nullptr,
                     ctx->mm_counters ? (uint32_t *)ctx->mm_counters->p : nullptr, E->d_Wd, E->d_idx, E->d_nnz, E->r};
    const uint32_t blocks = 8u * per_xcd;
    switch (act) {
    case SO_ACT_RELU:    return launch_quad<SO_ACT_RELU>(ctx, a, blocks);
    case SO_ACT_SIGMOID: return launch_quad<SO_ACT_SIGMOID>(ctx, a, blocks);
    case SO_ACT_TANH:    return launch_quad<SO_ACT_TANH>(ctx, a, blocks);
    default:             return launch_quad<SO_ACT_NONE>(ctx, a, blocks);
    }
}
