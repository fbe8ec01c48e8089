// Shared between the C-ABI front (api.hip) and the per-K kernel translation units
// (fused_kernel.hip compiled once per JABAS_K). Not part of the public interface.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>
#include "jabas_sync.h"

namespace jabas {

// Launch shape: threads per workgroup and tiles per workgroup (a tile = one 16-byte fp32 vector per
// thread; a chunk = consecutive tiles of a span, the share of one workgroup or, where that leaves compute
// units idle, of two or four: launch_split_log2). Small chunks keep the streamed window of every
// buffer compact (higher HBM rate) and cut the ramp-up / drain of a launch; kernels that carry many
// statistics have low occupancy and a long epilogue, and do better with more work per workgroup.
// Measured per kernel family (A/B builds of the whole library, every shape passes the parity suite):
//   full statistics rows          256 threads x 2 tiles (K <= 4) or 4 tiles (K > 4); 64, 128, 512 and
//                                 1024 threads were all slower (-2 ... -15 %)
//   similarity sums only          256 threads x 2 tiles: with four sums the K > 4 kernels fit 4 waves per SIMD
//                                 with two tiles of loads in flight
//   plain with optimizer, K > 4   256 threads x 2 tiles: +1 % over 512 x 1 and 512 x 2, +3 % over 256 x 4;
//                                 aggregate-only launches stay at 256 x 4
//   plain, Adam kinds, K <= 4     256 threads x 4 tiles, all loads of the chunk in flight at once: +0.5 ... +1.4 %
//                                 over 256 x 2 (8 tiles: -4 %)
//   plain, SGD, fp32, K <= 4      128 threads x 2 tiles: +2 ... +5 % over 256 x 2; 128 x 4 loses 5 % on the short
//                                 ResNet-50 launch when the buffers rotate out of the last-level cache (and reads
//                                 2 % faster than 128 x 2 when they do not: size sweeps over one buffer set mislead)
//   plain, everything else K <= 4 256 threads x 2 tiles
// (these figures are from after the planned launches began to read their tables through the constant address
// space; before that the plain K > 4 kernels were best at 512 x 1 and the K <= 4 ones at 2 tiles).
// The macros let a tuning build try other shapes without touching the sources.
#ifndef JABAS_BLOCK
#define JABAS_BLOCK 256
#endif
#ifndef JABAS_BLOCK_SGD
#define JABAS_BLOCK_SGD 128
#endif
#ifndef JABAS_BLOCK_MANYK
#define JABAS_BLOCK_MANYK 256
#endif
#ifndef JABAS_BLOCK_SIM_MANYK
#define JABAS_BLOCK_SIM_MANYK 256
#endif
#ifndef JABAS_CHUNK_TILES_LO
#define JABAS_CHUNK_TILES_LO 2
#endif
#ifndef JABAS_CHUNK_TILES_HI
#define JABAS_CHUNK_TILES_HI 4
#endif
#ifndef JABAS_CHUNK_TILES_MANYK
#define JABAS_CHUNK_TILES_MANYK 2
#endif
#ifndef JABAS_CHUNK_TILES_SIM_MANYK
#define JABAS_CHUNK_TILES_SIM_MANYK 2
#endif
#ifndef JABAS_CHUNK_TILES_SIM_LO
#define JABAS_CHUNK_TILES_SIM_LO JABAS_CHUNK_TILES_LO
#endif
#ifndef JABAS_CHUNK_TILES_PLAIN_LO
#define JABAS_CHUNK_TILES_PLAIN_LO 4
#endif
constexpr int kBlock = JABAS_BLOCK;         // default threads per workgroup (256 = 4 wave64)
constexpr int kWaves = kBlock / 64;
constexpr bool block_ok(int b) { return b % 64 == 0 && b >= 64 && b <= 1024; }
static_assert(block_ok(JABAS_BLOCK) && block_ok(JABAS_BLOCK_SGD) && block_ok(JABAS_BLOCK_MANYK) &&
              block_ok(JABAS_BLOCK_SIM_MANYK), "whole waves");
constexpr int kMinChunkTiles = JABAS_CHUNK_TILES_LO;
constexpr int kMaxChunkTiles = JABAS_CHUNK_TILES_HI;
// opt_class: 0 none, 1 SGD, 2 Adam/AdamW, 3 Adam/AdamW with amsgrad (launch shapes of class 2);
// stats: 0 none, 1 full rows, 2 similarity sums, 3 full rows + pair products (launch shapes and chunk
// tables of level 1). The shape depends
// on what a plan is encoded for (K, gradient dtype, optimizer class) and on the statistics level of the
// launch; a plan holds one chunk table per shape, so it serves every step.
__host__ __device__ constexpr int launch_block(int K, int grad_dtype, int opt_class, int stats) {
    if (stats == 2 && K > 4) return JABAS_BLOCK_SIM_MANYK;
    if (stats || opt_class == 0) return kBlock;
    if (K > 4) return JABAS_BLOCK_MANYK;
    return (opt_class == 1 && grad_dtype == JABAS_F32) ? JABAS_BLOCK_SGD : kBlock;
}
__host__ __device__ constexpr int launch_chunk_tiles(int K, int /*grad_dtype*/, int opt_class, int stats) {
    if (stats == 2) return K > 4 ? JABAS_CHUNK_TILES_SIM_MANYK : JABAS_CHUNK_TILES_SIM_LO;
    if (K > 4) return (stats || opt_class == 0) ? kMaxChunkTiles : JABAS_CHUNK_TILES_MANYK;
    if (!stats && opt_class >= 2) return JABAS_CHUNK_TILES_PLAIN_LO;
    return kMinChunkTiles;
}
// Statistics level whose launch shape (and chunk table of a plan) a level uses.
__host__ __device__ constexpr int shape_level(int stats) { return stats == JABAS_STATS_GRAM ? JABAS_STATS_FULL : stats; }
// log2 of the workgroups that share a chunk of a launch of n_chunks chunks, live(s) of them with a tile to work on at split s: a
// plan's tables know whole chunks only, the launch decides how many workgroups each of them gets. All figures: spans of one
// parameter group by value (unless stated) over buffers that rotate through more than the last-level cache; one set of buffers
// that stays there misleads.
//   short launches      below about 400 workgroups compute units idle and a workgroup takes its tiles in turn, each at the latency
//                       of memory. Whole chunks -> split: fp32 K = 4 AdamW 0.1 / 0.5 / 1.5 M elements 7.4 / 8.2 / 13.0 -> 4.1 / 6.0 /
//                       10.6 us, bf16 K = 8 AdamW full rows 0.1 / 0.5 M 12.0 / 13.1 -> 7.8 / 10.2. Split while there are fewer than
//                       2048 without statistics, 1 to 4 M elements lose: K = 4 AdamW 2 / 3 / 4 M 17.9 / 25.1 / 32.7 -> 19.0 / 27.5 /
//                       35.8, K = 8 bf16 aggregate 4 M 15.4 -> 18.0; while fewer than 512, 2 M 18.9, and K = 8 pair products 0.9 M
//                       0.90 of the time of whole chunks against 0.74
//   group changes       in a span (norms and biases between the weights): up to 512 with statistics; without, up to 2048, or 640 where a
//                       chunk is 1024 elements (SGD of up to four fp32 workers), whose halves are one tile of two waves.
//                       640 -> 2048 for the others, a change every 40000 elements, time in us: K = 1 fp32 amsgrad 1.7 / 4.5 / 6.5 M 14.3 / 32.5 /
//                       44.3 -> 13.4 / 30.7 / 42.1, K = 4 AdamW 3 / 4.5 / 6.5 M 25.7 / 37.7 / 52.9 -> 25.2 / 35.5 / 49.8, K = 3 bf16 AdamW 6.5 M
//                       42.0 -> 39.8; 1.4 M loses (K = 1 / 4 AdamW 9.5 / 13.5 -> 9.8 / 13.9); the same on buffers that stay in the
//                       last-level cache. SGD would lose with 2048: K = 2 fp32 1 M 6.8 -> 7.6, K = 1 5.8 -> 6.1, longer ones the same
//   without a tile      at most a quarter, or 64 with statistics (each still runs its epilogue and writes a row) and 256 without, or as
//                       many as there are compute units for: plans over short spans, one per small tensor, whose last chunk is
//                       mostly their only one. All splits -> these: 500 spans of 700 elements, K = 1 AdamW 7.7 -> 4.4 us, 20000, K = 16
//                       bf16 full rows 651 -> 502 (193 with the finalize of short spans)
//   full rows, K > 8    two workgroups per chunk at any size: these kernels hold one tile in flight and two or three waves per
//                       SIMD, and half the work per workgroup keeps the streamed window compact and the last round of
//                       workgroups short: ResNet-50 K = 16 bf16 254 -> 231 us (four: 240), 25 M elements K = 12 fp32 SGD
//                       302 -> 284, K = 16 fp32 AdamW 406 -> 390. Not bf16 gradients without an optimizer, whose reads alone are
//                       at the rate of memory: K = 12 / 16, 25 M 102 / 138 -> 113 / 162. K = 5..8 would gain 2-3 % with full
//                       rows and lose 11-14 % with pair products (25..40 sums per workgroup), and both levels cut their sums alike
//   with an optimizer,  the same for the same reason (one tile in flight, a chunk of two tiles) without statistics from 2048 chunks
//   K > 8               and with similarity sums from 4096 on, whether or not the group changes; where it does, plain launches are split
//                       below 2048 too, by the rule above, so that whole chunks are left to spans of one group of 448 to 2047 and to similarity
//                       sums of 512 to 4095. Engine steps of 100 tensors, whole chunks -> two workgroups each, fp32 K = 9 /
//                       12 / 16 AdamW with an aggregate, 6 M elements 67 / 80 / 98 -> 65 / 77 / 95 us, 20 M 216 / 259 / 319 -> 210 / 253 / 314,
//                       K = 16 SGD 100 M 1500 -> 1440; bf16 K = 16 AdamW amsgrad 40 M 463 -> 446; similarity sums, K = 12 fp32 SGD 20 M
//                       248 -> 240, bf16 K = 16 SGD 40 M 365 -> 353. Below, bf16 similarity sums lose up to 4 % (6 M, AdamW 68.5 -> 70.5)
//                       and plain launches of 3 M gain nothing
#ifndef JABAS_SPLIT_FROM_PLAIN
#define JABAS_SPLIT_FROM_PLAIN 2048
#endif
#ifndef JABAS_SPLIT_FROM_SIM
#define JABAS_SPLIT_FROM_SIM 4096
#endif
#ifndef JABAS_SPLIT_BELOW
#define JABAS_SPLIT_BELOW 448
#endif
#ifndef JABAS_SPLIT_BELOW_STATS
#define JABAS_SPLIT_BELOW_STATS 384
#endif
#ifndef JABAS_SPLIT_BELOW_GROUPS
#define JABAS_SPLIT_BELOW_GROUPS 2048
#endif
#ifndef JABAS_SPLIT_BELOW_GROUPS_SHORT
#define JABAS_SPLIT_BELOW_GROUPS_SHORT 640
#endif
#ifndef JABAS_SPLIT_BELOW_GROUPS_STATS
#define JABAS_SPLIT_BELOW_GROUPS_STATS 512
#endif
template <class Live>
inline uint32_t launch_split_log2(int K, int grad_dtype, int opt_class, int stats, uint64_t n_chunks, bool group_changes, const Live& live) {
    const uint32_t tiles = static_cast<uint32_t>(launch_chunk_tiles(K, grad_dtype, opt_class, stats));
    const bool short_chunks = 4 * static_cast<uint32_t>(launch_block(K, grad_dtype, opt_class, stats)) * tiles <= 1024;
    const uint64_t below = group_changes ? (stats ? JABAS_SPLIT_BELOW_GROUPS_STATS : short_chunks ? JABAS_SPLIT_BELOW_GROUPS_SHORT : JABAS_SPLIT_BELOW_GROUPS)
                                         : (stats ? JABAS_SPLIT_BELOW_STATS : JABAS_SPLIT_BELOW);
    const uint64_t empty = stats ? 64 : 256;
    const auto pays = [&](uint32_t s) {
        const uint64_t idle = (n_chunks << s) - live(s);
        return (n_chunks << s) <= 256 || idle <= empty || 3 * idle <= live(s);
    };
    const bool rows = stats == JABAS_STATS_FULL && (opt_class != 0 || grad_dtype == JABAS_F32);
    const bool long_step = opt_class != 0 && ((stats == JABAS_STATS_NONE && n_chunks >= JABAS_SPLIT_FROM_PLAIN) ||
                                              (stats == JABAS_STATS_SIMILARITY && n_chunks >= JABAS_SPLIT_FROM_SIM));
    uint32_t s = K > 8 && (rows || long_step) && pays(1) ? 1 : 0;
    while ((2u << s) <= tiles && live(s) < below && pays(s + 1)) ++s;
    return s;
}
// Width of the partial rows of a launch: 4 similarity sums, + K norms, + K(K-1)/2 pair products.
__host__ __device__ constexpr int stats_row_width(int K, int stats) {
    return stats == JABAS_STATS_FULL ? 4 + K : (stats == JABAS_STATS_GRAM ? 4 + K + K * (K - 1) / 2 : (stats ? 4 : 1));
}
// Widest rows of the statistics levels that are launched in the same chunks as `stats`: whether a launch is split further is
// asked of scratch for these, so that levels with sums in common cut them alike on any scratch and keep the same bits.
inline int shared_row_width(int K, int grad_dtype, int opt_class, int stats) {
    int width = 0;
    for (int level = JABAS_STATS_FULL; level <= JABAS_STATS_GRAM; ++level) {
        if (level == JABAS_STATS_GRAM && K > JABAS_STATS_GRAM_MAX_K) continue;
        if (launch_block(K, grad_dtype, opt_class, level) == launch_block(K, grad_dtype, opt_class, stats) &&
            launch_chunk_tiles(K, grad_dtype, opt_class, level) == launch_chunk_tiles(K, grad_dtype, opt_class, stats) &&
            stats_row_width(K, level) > width)
            width = stats_row_width(K, level);
    }
    return width;
}
constexpr int imin(int a, int b) { return a < b ? a : b; }
// Fewest elements a chunk of a launch with statistics covers: one partial row per chunk at least, sizes the static scratch, in
// which only launches short enough to leave room are split.
constexpr int kMinStatsChunkElems = 4 * imin(imin(JABAS_BLOCK * JABAS_CHUNK_TILES_LO, JABAS_BLOCK * JABAS_CHUNK_TILES_SIM_LO),
                                             JABAS_BLOCK_SIM_MANYK * JABAS_CHUNK_TILES_SIM_MANYK);
// Fewest elements any chunk covers, over all shapes: sizes blobs that must fit every launch, and workspaces (a tile of a launch
// with statistics, the least its workgroups take, is as long).
constexpr int kMinChunkElems = imin(imin(kMinStatsChunkElems, 4 * JABAS_BLOCK_SGD * JABAS_CHUNK_TILES_LO),
                                    4 * imin(imin(JABAS_BLOCK * JABAS_CHUNK_TILES_PLAIN_LO, JABAS_BLOCK * JABAS_CHUNK_TILES_LO),
                                             imin(JABAS_BLOCK_MANYK * JABAS_CHUNK_TILES_MANYK, JABAS_BLOCK * JABAS_CHUNK_TILES_HI)));
constexpr int kStatsStride = JABAS_STATS_STRIDE;
static_assert(stats_row_width(JABAS_STATS_GRAM_MAX_K, JABAS_STATS_GRAM) <= JABAS_STATS_STRIDE &&
              stats_row_width(JABAS_MAX_K, JABAS_STATS_FULL) <= JABAS_STATS_STRIDE, "every row fits the stride");

// Elements one thread handles per tile: one 16-byte fp32 vector of every fp32 buffer
// (bf16 gradients are then read as 8-byte vectors, which keeps every access of a wave
// contiguous).
__host__ __device__ constexpr int ept_of(int /*grad_dtype*/) { return 4; }
__host__ __device__ constexpr int tile_elems_of(int block) { return block * 4; }

// A span as the kernels see it. Pointers are rebased downwards by `lo` elements so that
// element index 0 of every buffer is 16-byte aligned (256-byte aligned when the buffers allow
// it, lo < 64 then, else lo < 4); [lo, hi) is the live range. Nothing below `lo` is accessed.
// Loose fp32 gradients (JABAS_SPAN_LOOSE_GRADS), and an aggregate in one of them, are 4-byte aligned only.
struct SpanDev {
    const void* g[JABAS_MAX_K];
    float* out;
    float* p;
    float* s1;
    float* s2;
    float* s3;
    float* fan[JABAS_MAX_K - 1];
    uint64_t lo, hi;
    // Where the Adam moments of grid element e live: float index mom(e) = t + mom_mult * (t & mom_mask),
    // t = e + mom_add, from s1 / s2 / s3. Arrays of their own: all three zero, mom(e) = e. Interleaved in
    // blocks of T elements: s1 = start of the span's first block group, s2 = s1 + T, s3 = s1 + 2 T,
    // mom_add = position of the first live element in its block minus lo (wraps; t >= 0 for every live e),
    // mom_mask = ~(T - 1), mom_mult = arrays interleaved - 1.
    uint64_t mom_add, mom_mask;
    uint32_t mom_mult;
    uint32_t narrow_ok;                      // 32-bit byte offsets reach every access of the span
    uint32_t n_fan;
    uint32_t bound_begin;
    uint32_t bound_count;
    uint32_t pad;
};
// Largest element index a 32-bit byte offset reaches in an fp32 buffer.
constexpr uint64_t kNarrowElems = 1ull << 30;

struct BoundDev {                            // same layout as JabasBound
    uint64_t start;                          // in un-rebased span coordinates
    uint32_t group;
    uint32_t pad;
};

// fp32 constants of one parameter group, derived on the host in double and rounded once,
// the way a Python float becomes an fp32 kernel scalar.
struct GroupDev {
    float wd;            // weight_decay
    float neg_lr;        // SGD: -lr
    float decay;         // AdamW: 1 - lr*wd
    float neg_step_size; // Adam: -(lr / (1 - beta1^t))
    float sqrt_bc2;      // Adam: sqrt(1 - beta2^t)
    float pad[3];
};

struct OptDev {
    float momentum, one_minus_damp;
    float beta1, one_minus_beta1, beta2, one_minus_beta2, eps;
    int32_t has_momentum, first_step, nesterov, adamw;
};

// chunk_tiles consecutive tiles of one span of a planned launch.
struct ChunkDesc {
    uint32_t span;                           // index into the span table
    uint32_t tile0;                          // first tile, local to the span
    uint32_t bound0;                         // bound entry (local to the span) covering the chunk's first live element
    uint32_t pad;
};

struct KArgs {
    const SpanDev* spans;                    // device table (planned launch)
    const ChunkDesc* chunks;                 // one per 2^split_log2 workgroups (planned launch)
    const uint32_t* chunk_prefix;            // n_span + 1 entries: first chunk of each span (planned launch)
    const BoundDev* bounds;                  // device, may be NULL
    double* partials;                        // one row of the level's width per workgroup
    const float* grad_scale;                 // device scalar or NULL (clipping)
    uint32_t n_span;
    uint32_t n_chunks;
    uint32_t chunk_tiles;                    // tiles per chunk (the kernel's own shape; checked on the host)
    uint32_t use_inline;                     // 1: the only span is `span0`, workgroup b starts at tile b * (chunk_tiles >> split_log2)
    uint32_t half_mask;                      // bit k set: VSW k belongs to half B
    uint32_t split_log2;                     // 2^split_log2 workgroups share a chunk (launch_split_log2)
    uint32_t writes_agg;                     // 1: a span's aggregate is written (the host's choice of residency; no kernel reads it)
    uint32_t pad;
    SpanDev span0;
    float w[JABAS_MAX_K];
    float wh[JABAS_MAX_K];
    OptDev opt;
    GroupDev groups[JABAS_MAX_GROUPS];
    const struct StepScal* dyn;              // device block holding this step's scalars, or NULL (they are the fields above)
};

// The scalars of a step that change from one step to the next (weights, optimizer constants, per-group
// constants), as a block in device memory: a launch that names such a block reads them from there instead
// of from its own arguments, so a launch recorded in a HIP graph can be replayed with the learning rate,
// the Adam step or the weights of the moment. Same layout on host and device; written by
// jabas_step_scalars_encode.
struct StepScal {
    float w[JABAS_MAX_K];
    float wh[JABAS_MAX_K];
    OptDev opt;
    uint32_t half_mask;
    GroupDev groups[JABAS_MAX_GROUPS];
};
static_assert(sizeof(StepScal) == JABAS_STEP_SCALARS_BYTES, "public size of the step-scalar block");

#if defined(__HIPCC__)
// Launch through hipLaunchKernel so that the status is the one of THIS launch: hipGetLastError() would
// also hand back (and clear) whatever an earlier, unrelated HIP call of the calling thread left behind.
template <typename... Params, typename... Given>
inline hipError_t launch_kernel(void (*kernel)(Params...), dim3 grid, dim3 block, size_t lds_bytes, hipStream_t stream,
                                Given&&... given) {
    static_assert(sizeof...(Params) == sizeof...(Given), "one argument per kernel parameter");
    std::tuple<Params...> values(static_cast<Params>(given)...);
    void* ptrs[sizeof...(Params) > 0 ? sizeof...(Params) : 1];
    std::apply([&](auto&... v) { size_t i = 0; ((ptrs[i++] = static_cast<void*>(&v)), ...); }, values);
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, lds_bytes, stream);
}

// Sum over the 64 lanes of a wave with DPP moves (no LDS traffic); the total lands in
// lane 63. Pairing order is fixed: lane^1, lane^2, mirror within 8, mirror within 16,
// row 0->1 and 2->3, rows 0..1 -> 2..3.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_move(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROW_MASK, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROW_MASK, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum_to_lane63(double v) {
    v += dpp_move<0xB1, 0xf>(v);    // quad_perm [1,0,3,2]
    v += dpp_move<0x4E, 0xf>(v);    // quad_perm [2,3,0,1]
    v += dpp_move<0x141, 0xf>(v);   // row_half_mirror
    v += dpp_move<0x140, 0xf>(v);   // row_mirror
    v += dpp_move<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    v += dpp_move<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
    return v;
}

#endif

// Per-K launchers, one translation unit each (fused_kernel.hip with -DJABAS_K=k).
// opt_class: 0 none, 1 SGD, 2 Adam/AdamW, 3 the same with amsgrad; dyn: the step's scalars come from a.dyn
// (classes 1 and 2 only).
// Returns hipError_t as int.
#define JABAS_DECLARE_K(k)                                                                   \
    int launch_fused_k##k(int grad_dtype, int opt_class, int stats, int dyn, const KArgs& a, \
                          unsigned grid, hipStream_t stream);
JABAS_DECLARE_K(1) JABAS_DECLARE_K(2) JABAS_DECLARE_K(3) JABAS_DECLARE_K(4)
JABAS_DECLARE_K(5) JABAS_DECLARE_K(6) JABAS_DECLARE_K(7) JABAS_DECLARE_K(8)
JABAS_DECLARE_K(9) JABAS_DECLARE_K(10) JABAS_DECLARE_K(11) JABAS_DECLARE_K(12)
JABAS_DECLARE_K(13) JABAS_DECLARE_K(14) JABAS_DECLARE_K(15) JABAS_DECLARE_K(16)
#undef JABAS_DECLARE_K

}  // namespace jabas
