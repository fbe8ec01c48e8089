// Fused VSW-aggregate + gradient statistics + optimizer kernel for gfx950 (MI355X).
// Compiled once per JABAS_K (number of virtual stream workers) so that the K gradient
// streams are fully unrolled into independent 128-bit loads.
//
// Execution shape
//   - one workgroup per chunk of consecutive tiles of one span, two or four where the launch is short or the kernel
//     holds one tile of many streams in flight (launch_split_log2); a tile is one 16-byte vector of
//     every fp32 buffer (one 8-byte vector of a bf16 gradient buffer) per thread. Threads per
//     workgroup and tiles per chunk depend on the kernel family (launch_block / launch_chunk_tiles):
//     256 threads x 2 or 4 tiles with statistics, 128 x 2, 256 x 2 or 256 x 4 without. Small,
//     short-lived workgroups dispatched in order keep the part of every buffer that is being
//     streamed at any moment compact, which on MI355X sustains a markedly higher HBM rate than a
//     persistent grid that spreads over the whole buffers;
//   - every global access is a vector access with the nontemporal hint (each byte is touched
//     exactly once per step);
//   - tiles that lie wholly inside the live range of a span take the vector path (all loads of U tiles issued
//     before any arithmetic, the parameter group looked up while they are under way); a tile that straddles a span
//     end, or is the only one left, goes wave by wave (single_tile), as do all of eight fp32 workers with pair products;
//   - statistics: per-thread fp64 accumulators -> LDS -> 16-way sums in fixed order -> DPP row
//     reduction -> one partial row of 4 + K doubles per workgroup in the workspace, summed in
//     fixed order by the finalize kernel. The order is fixed, so results are bit-identical run to run.
//
// Arithmetic is compiled with -ffp-contract=off: every fp32 product and sum of the
// aggregate and of the optimizer formulas is rounded on its own, so results can be
// compared bit for bit with a CPU restatement that applies the same operations in the
// same order. The formulas follow torch 1.8.1 optim/_functional.py (sgd, adam, adamw),
// the version the reference pins (README.md:59-64 of the JABAS repository).
#include "jabas_internal.h"

#ifndef JABAS_K
#error "compile with -DJABAS_K=<1..16>"
#endif
// Most tiles whose loads are in flight together: a whole 4-tile chunk without statistics,
// 2 tiles with (the fp64 accumulators need the registers).
#ifndef JABAS_UNROLL_PLAIN
#define JABAS_UNROLL_PLAIN 4
#endif
#ifndef JABAS_UNROLL_STATS
#define JABAS_UNROLL_STATS 2
#endif

namespace jabas {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
// fp32 gradients and the aggregate may sit at any element (JABAS_SPAN_LOOSE_GRADS). The access is the same instruction, which takes
// any multiple of 4 bytes; a wave whose vectors straddle lines touches nine of 128 bytes instead of eight. ShardAdamW.step over
// gradients packed at odd elements, an aligned copy of each such tensor before -> now: 1 M elements in 100 tensors 310 -> 50 us (then
// bound by its host side), 25.6 M in 60 219 -> 124, 80 M in 150 656 -> 385, 3 % over the rate of a copy.
typedef f32x4 __attribute__((aligned(4))) f32x4_a4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bits_to_float(uint32_t u) { return __builtin_bit_cast(float, u); }

// Address of element e of a buffer whose base is uniform over the workgroup. NARROW: the byte offset
// fits 32 bits (spans of up to kNarrowElems elements), so the address is "scalar base + zero-extended
// 32-bit lane offset": the form a global access takes with the base in scalar registers and ONE vector
// register of offset shared by every stream of the same element size, instead of a 64-bit vector
// address (two registers and two additions) per stream and tile.
template <bool NARROW, int ES> __device__ __forceinline__ const char* elem_addr(const void* base, uint64_t e) {
    if constexpr (NARROW) {
        const uint32_t off = static_cast<uint32_t>(e) * static_cast<uint32_t>(ES);
        return static_cast<const char*>(base) + static_cast<uint64_t>(off);
    } else {
        return static_cast<const char*>(base) + e * ES;
    }
}

template <int DT> struct Grad;

template <> struct Grad<JABAS_F32> {
    using Raw = f32x4;
    using Mem = f32x4_a4;
    template <bool NARROW> static __device__ __forceinline__ Raw load(const void* base, uint64_t e) {
        return __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4*>(elem_addr<NARROW, 4>(base, e)));
    }
    static __device__ __forceinline__ float elem(const Raw& r, int i) { return r[i]; }
    // elements at byte addresses of one stream, the live ones of a vector that straddles a span end
    static __device__ __forceinline__ Raw gather(const char* const (&at)[4], const bool (&live)[4]) {
        Raw r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = *reinterpret_cast<const float*>(at[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = live[i] ? r[i] : 0.0f;
        return r;
    }
};

template <> struct Grad<JABAS_BF16> {
    using Raw = u32x2;
    using Mem = u32x2;
    template <bool NARROW> static __device__ __forceinline__ Raw load(const void* base, uint64_t e) {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(elem_addr<NARROW, 2>(base, e)));
    }
    // bf16 -> fp32 is exact: the 16 bits become the high half of the fp32 pattern.
    static __device__ __forceinline__ float elem(const Raw& r, int i) {
        const uint32_t w = i < 2 ? r.x : r.y;
        return bits_to_float(i & 1 ? w & 0xffff0000u : w << 16);
    }
    static __device__ __forceinline__ Raw gather(const char* const (&at)[4], const bool (&live)[4]) {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = *reinterpret_cast<const uint16_t*>(at[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = live[i] ? h[i] : 0u;
        return Raw{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
};

constexpr int OPT_NONE = 0, OPT_SGD = 1, OPT_ADAM = 2, OPT_AMS = 3;    // OPT_AMS: Adam / AdamW with amsgrad
__host__ __device__ constexpr bool is_adam(int opt) { return opt == OPT_ADAM || opt == OPT_AMS; }
// Kernels with statistics form the addresses of the vector path as scalar base + 32-bit lane offset (measured
// on the ViT-L/16 set, K = 8 bf16: +0.5 % with full rows, +2 % with similarity sums; K = 4 fp32 Adam: 8-9 fewer
// VGPRs, full rows 131 -> 123 and 4 waves per SIMD instead of 3, ViT-B/16 +1.2 % with similarity sums, +0.4 % with
// full rows, GNMT +-0.3 %); their spans that 32-bit byte offsets do not reach (over 4 GiB of fp32 per buffer)
// go tile by tile (single_tile): correct but slower. The plain kernels keep 64-bit vector addresses
// (no gain there: their registers are not what limits them).
__host__ __device__ constexpr bool narrow_addressing(int /*K*/, int SL) { return SL != 0; }

// Statistics level of a launch: 0 none, 1 the full row (4 + K sums), 2 the four sums of the halves and of
// the aggregate only (what the cosine similarity and global-norm clipping read), 3 the full row and the
// products of every pair of workers (the Gram matrix; up to JABAS_STATS_GRAM_MAX_K workers).
template <int K, int SL> struct NStats { static constexpr int value = stats_row_width(K, SL); };
constexpr bool per_vsw_norms(int SL) { return SL == JABAS_STATS_FULL || SL == JABAS_STATS_GRAM; }

// Per-thread running sums of the statistics. fp32 gradients: fp64 (a product of two fp32 values is exact
// in fp64). bf16 gradients: fp32 within the thread's chunk (at most 16 elements), widened to fp64 when the
// workgroup reduces: a product of two bf16 values is exact in fp32 and the few fp32 additions keep the
// sums within 1e-6 relative, four orders inside the 1e-2 bar of reduced-precision gradients, at a third
// of the arithmetic and half the registers (fp64 multiply-adds and conversions run at half rate).
template <int DT> struct StatAcc { using type = double; };
template <> struct StatAcc<JABAS_BF16> { using type = float; };
__device__ __forceinline__ double stat_fma(float a, float b, double acc) {
    return __builtin_fma(static_cast<double>(a), static_cast<double>(b), acc);
}
__device__ __forceinline__ float stat_fma(float a, float b, float acc) { return __builtin_fmaf(a, b, acc); }

// The step's scalars as the arithmetic below names them (a.w[k], a.wh[k], a.half_mask, a.opt, a.groups[i],
// plus a.bounds and a.grad_scale), backed by a StepScal block in device memory instead of the kernel
// arguments. The block is read through the constant address space: uniform loads that the compiler may
// place anywhere, the same instructions a kernel-argument read compiles to, and the block is not written
// while a launch that names it runs. Every function below takes either KArgs or this view.
struct DynView {
    typedef const __attribute__((address_space(4))) StepScal* Block;
    struct Weights {
        const __attribute__((address_space(4))) float* p;
        __device__ __forceinline__ float operator[](int k) const { return p[k]; }
    };
    struct Groups {
        Block b;
        __device__ __forceinline__ GroupDev operator[](uint32_t i) const {
            GroupDev g;
            g.wd = b->groups[i].wd; g.neg_lr = b->groups[i].neg_lr; g.decay = b->groups[i].decay;
            g.neg_step_size = b->groups[i].neg_step_size; g.sqrt_bc2 = b->groups[i].sqrt_bc2;
            return g;
        }
    };
    Weights w, wh;
    Groups groups;
    OptDev opt;
    uint32_t half_mask;
    const BoundDev* bounds;
    const float* grad_scale;
    __device__ __forceinline__ explicit DynView(const KArgs& a) {
        Block b = (Block)a.dyn;
        w.p = b->w; wh.p = b->wh; groups.b = b;
        opt.momentum = b->opt.momentum; opt.one_minus_damp = b->opt.one_minus_damp;
        opt.beta1 = b->opt.beta1; opt.one_minus_beta1 = b->opt.one_minus_beta1;
        opt.beta2 = b->opt.beta2; opt.one_minus_beta2 = b->opt.one_minus_beta2; opt.eps = b->opt.eps;
        opt.has_momentum = b->opt.has_momentum; opt.first_step = b->opt.first_step;
        opt.nesterov = b->opt.nesterov; opt.adamw = b->opt.adamw;
        half_mask = b->half_mask;
        bounds = a.bounds;
        grad_scale = a.grad_scale;
    }
};

// The bound table of a launch is, like the plan's other tables, not written while the launch runs: read through
// the constant address space (uniform loads the compiler is free to move or repeat).
typedef const __attribute__((address_space(4))) BoundDev* ConstBounds;
__device__ __forceinline__ ConstBounds const_bounds(const BoundDev* p) { return (ConstBounds)p; }

// Float index of grid element e's Adam moments from the span's moment bases: e itself when the moments are
// arrays of their own, its place in the interleaved arena otherwise (SpanDev). Two integer operations.
template <class SP> __device__ __forceinline__ uint64_t moment_index(const SP& sp, uint64_t e) {
    const uint64_t t = e + sp.mom_add;
    return t + sp.mom_mult * (t & sp.mom_mask);
}

// One element of the optimizer step. g is the aggregated gradient.
template <int OPT>
__device__ __forceinline__ void opt_elem(float g, float& p, float& s1, float& s2, float& s3,
                                         const GroupDev& G, const OptDev& O) {
    if constexpr (OPT == OPT_SGD) {
        float d = g;
        if (G.wd != 0.0f) d = d + G.wd * p;
        if (O.has_momentum) {
            if (O.first_step) s1 = d;
            else s1 = s1 * O.momentum + d * O.one_minus_damp;
            d = O.nesterov ? d + O.momentum * s1 : s1;
        }
        p = p + G.neg_lr * d;
    } else if constexpr (is_adam(OPT)) {
        if (O.adamw) p = p * G.decay;
        else if (G.wd != 0.0f) g = g + G.wd * p;
        s1 = s1 * O.beta1 + g * O.one_minus_beta1;
        s2 = s2 * O.beta2 + (O.one_minus_beta2 * g) * g;
        float second = s2;
        if constexpr (OPT == OPT_AMS) {       // torch.maximum(max_exp_avg_sq, exp_avg_sq): a NaN on either side stays
            s3 = (s3 != s3) ? s3 : ((s2 != s2) ? s2 : (s3 > s2 ? s3 : s2));
            second = s3;
        }
        const float denom = __builtin_sqrtf(second) / G.sqrt_bc2 + O.eps;
        p = p + (G.neg_step_size * s1) / denom;
    }
}

// Aggregate and statistics of a thread's four elements of a tile, out of the vectors as loaded. They are widened one element
// at a time: all four at once keep 4 K floats alive beside the vectors.
template <int K, int DT, int SL, bool HD, class A>
__device__ __forceinline__ void aggregate(const typename Grad<DT>::Raw (&raw)[K], float (&agg)[4], const A& a, float clip,
                                          typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float g[K];
#pragma unroll
        for (int k = 0; k < K; ++k) g[k] = Grad<DT>::elem(raw[k], i);
        float s = g[0] * a.w[0];
#pragma unroll
        for (int k = 1; k < K; ++k) s = s + g[k] * a.w[k];
        if (clip < 1.0f) s = s * clip;         // global-norm clipping: only ever scales down
        agg[i] = s;
        if constexpr (SL) {
            float ga = 0.0f, gb = 0.0f;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const float t = g[k] * a.wh[k];
                if constexpr (HD) {            // default halves: even worker -> A, odd -> B
                    if (k & 1) gb = gb + t; else ga = ga + t;
                } else {
                    const bool in_b = (a.half_mask >> k) & 1u;
                    gb = in_b ? gb + t : gb;
                    ga = in_b ? ga : ga + t;
                }
                if constexpr (per_vsw_norms(SL))
                    acc[JABAS_STAT_NORM_VSW0 + k] = stat_fma(g[k], g[k], acc[JABAS_STAT_NORM_VSW0 + k]);
                if constexpr (SL == JABAS_STATS_GRAM) {
#pragma unroll
                    for (int b = k + 1; b < K; ++b)
                        acc[JABAS_STAT_PAIR(K, k, b)] = stat_fma(g[k], g[b], acc[JABAS_STAT_PAIR(K, k, b)]);
                }
            }
            // fp64 sums: fp32 x fp32 products are exact in fp64, so fma == mul followed by add there.
            acc[JABAS_STAT_DOT_AB] = stat_fma(ga, gb, acc[JABAS_STAT_DOT_AB]);
            acc[JABAS_STAT_NORM_A] = stat_fma(ga, ga, acc[JABAS_STAT_NORM_A]);
            acc[JABAS_STAT_NORM_B] = stat_fma(gb, gb, acc[JABAS_STAT_NORM_B]);
            acc[JABAS_STAT_NORM_AGG] = stat_fma(s, s, acc[JABAS_STAT_NORM_AGG]);
            // keep the elements' dependency chains apart: interleaving them costs the statistics
            // kernels a third of their occupancy in registers and buys nothing in a memory-bound loop
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The parameter group a wave is in, in scalar registers: entry j of the span's bound table, which ends at element `end` of the
// span. Looked up while the loads of the wave's elements are under way, not before they are issued: a table read is a trip to
// memory for the first waves of a launch.
template <bool SEARCH> struct GroupCursor {
    ConstBounds bd;
    uint32_t nb, j;
    uint64_t end;                                // 0: not looked up yet
    uint32_t group;                              // of entry j
    uint32_t id;                                 // the group whose constants g holds, JABAS_MAX_GROUPS at first
    GroupDev g;
    __device__ __forceinline__ void look_up() {
        group = nb ? bd[j].group & (JABAS_MAX_GROUPS - 1) : 0;           // a bound table on the device cannot be checked by the host
        end = j + 1 < nb ? bd[j + 1].start : ~static_cast<uint64_t>(0);
    }
    // moves on to the entry of element rel >= end. SEARCH: j is not known to be near (a span by value has no chunk table).
    __device__ __forceinline__ void seek(uint64_t rel) {
        if (SEARCH && end == 0) {                // largest j with bd[j].start <= rel
            uint32_t lo = 0, hi = nb;
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (bd[mid].start <= rel) lo = mid; else hi = mid;
            }
            j = lo;
        }
        while (j + 1 < nb && bd[j + 1].start <= rel) ++j;
        look_up();
    }
    // The groups of a thread's four elements, a byte each, of a wave's share that begins at element rel0 in entry j and ends before
    // rel_end in a later entry, which becomes j. named: all groups of the share, a bit each.
    __device__ __forceinline__ uint32_t groups_of_thread(uint64_t rel0, uint64_t rel_end, uint32_t& named) {
        const int lane4 = static_cast<int>(threadIdx.x & 63) * 4;
        uint32_t ids = group * 0x01010101u;
        do {
            const int before = static_cast<int>(end - rel0) - lane4;     // of the thread's elements, before the entry
            const uint32_t keep = static_cast<uint32_t>((1ull << (8 * (before < 0 ? 0 : before > 4 ? 4 : before))) - 1);
            ++j;
            look_up();
            ids = (ids & keep) | (group * 0x01010101u & ~keep);
            named |= 1u << group;
        } while (end < rel_end);
        return ids;
    }
};

constexpr uint32_t kWaveElems = 256;             // of a tile: 64 lanes, four elements each

// Whether elements of another group are jumped over, a branch per element, instead of going through the arithmetic and keeping
// their values. That takes 5 to 15 registers less and 1 to 2.5 % more time (K = 1 Adam 160 M elements 717 -> 737 us; K = 5 and 6 bf16
// with statistics, 40 M, 1 %), so only where it decides between one wave per SIMD and two: amsgrad with the pair products of eight
// fp32 workers, 263 -> 248 registers, 40 M elements 576 -> 474 us, without an aggregate 518 -> 436.
constexpr bool update_branches(int K, int DT, int OPT, int SL) {
    return OPT == OPT_AMS && SL == JABAS_STATS_GRAM && DT == JABAS_F32 && K > 7;
}

// Optimizer step on the live elements [first, last) of a wave's share of a tile, one pass per parameter group that the share names:
// almost always one. Elements of another group go through the arithmetic too and keep their values; BRANCH: they jump over it.
// rel0: the wave's first element, in span coordinates. What a dead element comes to is not stored.
// A pass per change instead, until the wave's share ends, made spans of tiny tensors slow. Two groups in turn, a pass per change -> per
// group: changes every 16 elements, 3 M, K = 4 AdamW similarity sums 107 -> 50 us, K = 1 AdamW 105 -> 44, K = 2 SGD 54 -> 43; every 100,
// 0.3 M, K = 4 AdamW 10.0 -> 7.8; one group within 1 %. A thread's entries read two or 64 at a time instead of one: K = 2 SGD 43 -> 38
// for a fifth more spilled scalar registers, or four vector registers more.
template <bool BRANCH, int OPT, int SL, class A, class C>
__device__ __forceinline__ void update(const float (&agg)[4], f32x4& p, f32x4& s1, f32x4& s2, f32x4& s3, const A& a, C& cur,
                                       uint64_t rel0, uint32_t first, uint32_t last) {
    if (rel0 + first >= cur.end) cur.seek(rel0 + first);
    uint32_t named = 1u << cur.group, ids = cur.group * 0x01010101u;
    if (cur.end < rel0 + last) ids = cur.groups_of_thread(rel0, rel0 + last, named);
    while (true) {
        const uint32_t id = static_cast<uint32_t>(__builtin_ctz(named));
        if (id != cur.id) {
            cur.id = id;
            cur.g = a.groups[id];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = (ids >> (8 * i) & 255u) == id;
            if (!BRANCH || in) {
                float np = p[i], n1 = s1[i], n2 = 0.0f, n3 = 0.0f;
                if constexpr (is_adam(OPT)) n2 = s2[i];
                if constexpr (OPT == OPT_AMS) n3 = s3[i];
                opt_elem<OPT>(agg[i], np, n1, n2, n3, cur.g, a.opt);
                p[i] = in ? np : p[i];
                s1[i] = in ? n1 : s1[i];
                if constexpr (is_adam(OPT)) s2[i] = in ? n2 : s2[i];
                if constexpr (OPT == OPT_AMS) s3[i] = in ? n3 : s3[i];
            }
            if constexpr (SL) __builtin_amdgcn_sched_barrier(0);
        }
        named &= named - 1;
        if (named == 0) return;
    }
}

template <bool NARROW> __device__ __forceinline__ f32x4 load_vec(const float* base, uint64_t e) {
    return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(elem_addr<NARROW, 4>(base, e)));
}
template <bool NARROW, class MEM = f32x4> __device__ __forceinline__ void store_vec(const f32x4& r, float* base, uint64_t e) {
    __builtin_nontemporal_store(r, reinterpret_cast<MEM*>(const_cast<char*>(elem_addr<NARROW, 4>(base, e))));
}

// Registers of U consecutive tiles: the raw vectors as loaded.
template <int K, int DT, int U, int OPT = OPT_ADAM> struct TileRegs {
    typename Grad<DT>::Raw g[U][K];
    f32x4 p[U], s1[U], s2[U], s3[OPT == OPT_AMS ? U : 1];
};

// Issues every load of U consecutive full tiles. e is the (rebased) index of this
// thread's first element in the first tile.
template <int K, int DT, int OPT, int U, int BS, bool NARROW, class SP>
__device__ __forceinline__ void issue_loads(TileRegs<K, DT, U, OPT>& r, const SP& sp, uint64_t e, bool load_s1) {
    constexpr uint64_t TE = static_cast<uint64_t>(BS) * 4;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint64_t eu = e + u * TE;
#pragma unroll
        for (int k = 0; k < K; ++k) r.g[u][k] = Grad<DT>::template load<NARROW>(sp.g[k], eu);
        if constexpr (OPT != OPT_NONE) {
            r.p[u] = load_vec<NARROW>(sp.p, eu);
            const uint64_t mu = is_adam(OPT) ? moment_index(sp, eu) : eu;
            r.s1[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (load_s1) r.s1[u] = load_vec<NARROW>(sp.s1, mu);
            if constexpr (is_adam(OPT)) r.s2[u] = load_vec<NARROW>(sp.s2, mu);
            if constexpr (OPT == OPT_AMS) r.s3[u] = load_vec<NARROW>(sp.s3, mu);
        }
    }
}

// Arithmetic and stores of U full tiles whose loads were issued by issue_loads.
template <int K, int DT, int OPT, int SL, bool HD, int U, bool NARROW, class A, class SP, class C>
__device__ __forceinline__ void consume(TileRegs<K, DT, U, OPT>& r, const SP& sp, uint64_t e, uint64_t rel0, const A& a, C& cur, float clip,
                                        bool use_s1, float* out, typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    constexpr uint64_t TE = static_cast<uint64_t>(launch_block(K, DT, OPT, SL)) * 4;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint64_t eu = e + u * TE;
        float agg[4];
        aggregate<K, DT, SL, HD>(r.g[u], agg, a, clip, acc);
        if (out) store_vec<NARROW, f32x4_a4>(f32x4{agg[0], agg[1], agg[2], agg[3]}, out, eu);
        if constexpr (OPT != OPT_NONE) {
            f32x4& s3 = r.s3[OPT == OPT_AMS ? u : 0];
            update<update_branches(K, DT, OPT, SL), OPT, SL>(agg, r.p[u], r.s1[u], r.s2[u], s3, a, cur, rel0 + u * TE, 0u, kWaveElems);
            store_vec<NARROW>(r.p[u], sp.p, eu);
            const uint64_t mu = is_adam(OPT) ? moment_index(sp, eu) : eu;
            if (use_s1) store_vec<NARROW>(r.s1[u], sp.s1, mu);
            if constexpr (is_adam(OPT)) store_vec<NARROW>(r.s2[u], sp.s2, mu);
            if constexpr (OPT == OPT_AMS) store_vec<NARROW>(s3, sp.s3, mu);
            for (uint32_t f = 0; f < sp.n_fan; ++f) store_vec<NARROW>(r.p[u], sp.fan[f], eu);
        }
    }
}

__device__ __forceinline__ uint32_t wave_of_workgroup() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Vector path over nfull consecutive full tiles: groups of U tiles, then U/2, ... down to LEAST. Returns the tiles left over.
template <int K, int DT, int OPT, int SL, bool HD, int U, int LEAST, class A, class SP, class C>
__device__ __forceinline__ uint32_t fast_run(const SP& sp, uint64_t e0, uint32_t nfull, const A& a, C& cur, float clip, bool use_s1, bool load_s1,
                                             float* out, typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    constexpr int BS = launch_block(K, DT, OPT, SL);
    constexpr uint64_t TE = static_cast<uint64_t>(BS) * 4;
    uint32_t i = 0;
    for (; i + U <= nfull; i += U, e0 += U * TE) {
        const uint64_t e = e0 + static_cast<uint64_t>(threadIdx.x) * 4;
        TileRegs<K, DT, U, OPT> r;
        issue_loads<K, DT, OPT, U, BS, narrow_addressing(K, SL)>(r, sp, e, load_s1);
        consume<K, DT, OPT, SL, HD, U, narrow_addressing(K, SL)>(r, sp, e, e0 - sp.lo + wave_of_workgroup() * kWaveElems, a, cur, clip, use_s1, out, acc);
    }
    if constexpr (U > LEAST) return fast_run<K, DT, OPT, SL, HD, U / 2, LEAST>(sp, e0, nfull - i, a, cur, clip, use_s1, load_s1, out, acc);
    else return nfull - i;
}

// Place of a wave's share of a tile in a span's streams: element `first`, its first live one, is the scalar base, a lane's
// elements lie `at` elements behind it and their moments `mom` (32 bits: any length of span).
struct WavePlace {
    uint64_t e, m;                               // grid index and moment index of the wave's first live element
    uint32_t first, last;                        // live elements, wave-relative
    template <class SP> __device__ __forceinline__ WavePlace(const SP& sp, uint64_t wave_e) {
        first = sp.lo > wave_e ? static_cast<uint32_t>(sp.lo - wave_e < kWaveElems ? sp.lo - wave_e : kWaveElems) : 0u;
        last = sp.hi > wave_e ? static_cast<uint32_t>(sp.hi - wave_e < kWaveElems ? sp.hi - wave_e : kWaveElems) : 0u;
        e = wave_e + first;
        m = moment_index(sp, e);
    }
    template <class SP> __device__ __forceinline__ uint32_t moment_at(const SP& sp, uint32_t at) const {
        const uint32_t t = static_cast<uint32_t>(e + sp.mom_add), mask = static_cast<uint32_t>(sp.mom_mask);
        return at + sp.mom_mult * (((t + at) & mask) - (t & mask));
    }
};
template <int ES> __device__ __forceinline__ const char* lane_addr(const void* base, uint64_t e, uint32_t at) {
    return static_cast<const char*>(base) + e * ES + static_cast<uint64_t>(at * ES);
}
__device__ __forceinline__ f32x4 load_at(const float* base, uint64_t e, uint32_t at) {
    return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(lane_addr<4>(base, e, at)));
}
__device__ __forceinline__ f32x4 gather_at(const float* base, uint64_t e, const uint32_t (&at)[4], const bool (&live)[4]) {
    const char* const p[4] = {lane_addr<4>(base, e, at[0]), lane_addr<4>(base, e, at[1]), lane_addr<4>(base, e, at[2]), lane_addr<4>(base, e, at[3])};
    return Grad<JABAS_F32>::gather(p, live);
}
template <class MEM = f32x4> __device__ __forceinline__ void store_at(const f32x4& r, float* base, uint64_t e, uint32_t at) {
    __builtin_nontemporal_store(r, reinterpret_cast<MEM*>(const_cast<char*>(lane_addr<4>(base, e, at))));
}

// One tile, wave by wave, wherever it lies in the span. A thread whose four elements are all live takes the vector accesses; the
// few that straddle the span's first or last element gather theirs, every load issued before any is waited for (indices of dead
// elements are those of live ones, their values zero: nothing outside the span is touched, the sums are not changed).
// A launch of a few hundred workgroups lasts as long as its slowest one. Before, a tile with a group change was taken by itself,
// each thread looking up its own bounds and those that straddled one working element by element, a trip to memory each: such a
// workgroup took 9 to 10 us where the others took 4 (K = 8 bf16 AdamW, similarity sums, 0.3 M elements), and the table was read
// before any load was issued. Sync launch alone, 46 to 60 tensors, before -> now in us:
//   K = 4 fp32 AdamW   0.3 M none 8.8 -> 6.2, similarity sums 10.6 -> 6.7   1.2 M 15.2 -> 13.2, 17.8 -> 14.2   5 M 40.8 -> 36.9, 42.3 -> 39.5
//   K = 8 bf16 AdamW   0.3 M none 9.0 -> 6.2, pair products 12.4 -> 9.6     1.2 M 15.6 -> 12.8, 23.1 -> 17.6   5 M 40.9 -> 38.1, 51.1 -> 45.2
//   K = 2 fp32 SGD     0.3 M none 5.6 -> 4.3, similarity sums 7.5 -> 5.3    1.2 M 10.8 -> 8.8, 13.9 -> 10.0    5 M 26.9 -> 24.7, 28.8 -> 26.3
// and 25 M the same within 2 %.
template <int K, int DT, int OPT, int SL, bool HD, class A, class SP, class C>
__device__ __forceinline__ void single_tile(const SP& sp, uint64_t tile_e0, const A& a, C& cur, float clip, bool use_s1, bool load_s1, float* out,
                                            typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    using GR = Grad<DT>;
    constexpr int GS = DT == JABAS_BF16 ? 2 : 4;
    const uint64_t wave_e = tile_e0 + wave_of_workgroup() * kWaveElems;
    const WavePlace w(sp, wave_e);
    if (w.first >= w.last) return;               // none of the wave's elements is live
    const uint32_t lane4 = (threadIdx.x & 63) * 4;
    const bool whole = lane4 >= w.first && lane4 + 4 <= w.last, some = lane4 + 4 > w.first && lane4 < w.last;
    const uint32_t at = lane4 - w.first, mom = w.moment_at(sp, at);
    uint32_t eat[4], emom[4];
    bool live[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        live[i] = lane4 + i >= w.first && lane4 + i < w.last;
        eat[i] = live[i] ? at + i : (lane4 + i < w.first ? 0u : w.last - 1 - w.first);
        emom[i] = w.moment_at(sp, eat[i]);
    }
    TileRegs<K, DT, 1, OPT> r;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    if (whole) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            r.g[0][k] = __builtin_nontemporal_load(reinterpret_cast<const typename GR::Mem*>(lane_addr<GS>(sp.g[k], w.e, at)));
        if constexpr (OPT != OPT_NONE) {
            r.p[0] = load_at(sp.p, w.e, at);
            r.s1[0] = zero;
            if (load_s1) r.s1[0] = is_adam(OPT) ? load_at(sp.s1, w.m, mom) : load_at(sp.s1, w.e, at);
            if constexpr (is_adam(OPT)) r.s2[0] = load_at(sp.s2, w.m, mom);
            if constexpr (OPT == OPT_AMS) r.s3[0] = load_at(sp.s3, w.m, mom);
        }
    } else if (some) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const char* const p[4] = {lane_addr<GS>(sp.g[k], w.e, eat[0]), lane_addr<GS>(sp.g[k], w.e, eat[1]),
                                      lane_addr<GS>(sp.g[k], w.e, eat[2]), lane_addr<GS>(sp.g[k], w.e, eat[3])};
            r.g[0][k] = GR::gather(p, live);
            if constexpr (K > 8) {               // a few workers at a time: sixteen streams of four elements would set the register count
                if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (OPT != OPT_NONE) {
            r.p[0] = gather_at(sp.p, w.e, eat, live);
            r.s1[0] = zero;
            if (load_s1) r.s1[0] = is_adam(OPT) ? gather_at(sp.s1, w.m, emom, live) : gather_at(sp.s1, w.e, eat, live);
            if constexpr (is_adam(OPT)) r.s2[0] = gather_at(sp.s2, w.m, emom, live);
            if constexpr (OPT == OPT_AMS) r.s3[0] = gather_at(sp.s3, w.m, emom, live);
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) r.g[0][k] = typename GR::Raw{};
        if constexpr (OPT != OPT_NONE) {
            r.p[0] = r.s1[0] = zero;
            if constexpr (is_adam(OPT)) r.s2[0] = zero;
            if constexpr (OPT == OPT_AMS) r.s3[0] = zero;
        }
    }
    float agg[4];
    aggregate<K, DT, SL, HD>(r.g[0], agg, a, clip, acc);
    if constexpr (OPT != OPT_NONE) update<update_branches(K, DT, OPT, SL), OPT, SL>(agg, r.p[0], r.s1[0], r.s2[0], r.s3[0], a, cur, wave_e - sp.lo, w.first, w.last);
    if (whole) {
        if (out) store_at<f32x4_a4>(f32x4{agg[0], agg[1], agg[2], agg[3]}, out, w.e, at);
        if constexpr (OPT != OPT_NONE) {
            store_at(r.p[0], sp.p, w.e, at);
            if (use_s1) { if constexpr (is_adam(OPT)) store_at(r.s1[0], sp.s1, w.m, mom); else store_at(r.s1[0], sp.s1, w.e, at); }
            if constexpr (is_adam(OPT)) store_at(r.s2[0], sp.s2, w.m, mom);
            if constexpr (OPT == OPT_AMS) store_at(r.s3[0], sp.s3, w.m, mom);
            for (uint32_t f = 0; f < sp.n_fan; ++f) store_at(r.p[0], sp.fan[f], w.e, at);
        }
    } else if (some) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!live[i]) continue;
            if (out) out[w.e + eat[i]] = agg[i];
            if constexpr (OPT != OPT_NONE) {
                sp.p[w.e + eat[i]] = r.p[0][i];
                if (use_s1) sp.s1[is_adam(OPT) ? w.m + emom[i] : w.e + eat[i]] = r.s1[0][i];
                if constexpr (is_adam(OPT)) sp.s2[w.m + emom[i]] = r.s2[0][i];
                if constexpr (OPT == OPT_AMS) sp.s3[w.m + emom[i]] = r.s3[0][i];
                for (uint32_t f = 0; f < sp.n_fan; ++f) sp.fan[f][w.e + eat[i]] = r.p[0][i];
            }
        }
    }
}

// Tiles [lt0, lt1) of one span (tile indices local to the span). SEARCH: no bound entry near their first element is known.
template <int K, int DT, int OPT, int SL, bool HD, bool SEARCH, class A, class SP>
__device__ __forceinline__ void span_range(const SP& sp, uint32_t lt0, uint32_t lt1, uint32_t j0,
                                           const A& a, typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    const float clip = a.grad_scale ? *a.grad_scale : 1.0f;      // uniform: one scalar load per workgroup
    // One fp32 worker of weight 1 whose aggregate is its own buffer, no clipping or a coefficient that scales nothing: the
    // buffer already holds what would be written, 4 of 24 (SGD) or 32 (Adam) bytes per element. That is the step of a
    // single VSW and the second launch of a clipped step whose norm stays under the bound (a worker's NaN keeps its bits).
    // 20 M elements SGD 82 -> 67 us, 80 M AdamW with similarity sums 425 -> 360; clipped AdamW of four, 20 M, norm under the
    // bound 182 -> 167, over it 182.
    float* out = sp.out;
    if constexpr (K == 1 && DT == JABAS_F32) {
        if (static_cast<const void*>(out) == sp.g[0] && a.w[0] == 1.0f && !(clip < 1.0f)) out = nullptr;
    }
    constexpr uint64_t TE = static_cast<uint64_t>(launch_block(K, DT, OPT, SL)) * 4;
    constexpr int UW = SL ? JABAS_UNROLL_STATS : JABAS_UNROLL_PLAIN;
    constexpr int CT = launch_chunk_tiles(K, DT, OPT, SL);
    constexpr int U0 = UW < CT ? UW : CT;     // never more than a chunk holds
    // 9..16 gradient streams: one tile's loads fill the registers; so do eight fp32 ones beside the 28 fp64 pair
    // sums of the Gram level (two tiles in flight: 256 registers and one wave per SIMD, 13 % slower)
    constexpr int U = (K > 8 || (SL == JABAS_STATS_GRAM && DT == JABAS_F32 && K > 7)) ? 1 : U0;
    constexpr int LEAST = U > 1 ? 2 : 1;      // a single tile goes through single_tile, unless it is all that is ever in flight
    static_assert((U & (U - 1)) == 0, "the unroll cascade halves U down to LEAST");
    const bool use_s1 = is_adam(OPT) || (OPT == OPT_SGD && a.opt.has_momentum);
    const bool load_s1 = is_adam(OPT) || (OPT == OPT_SGD && a.opt.has_momentum && !a.opt.first_step);
    const uint32_t nb = sp.bound_count;
    GroupCursor<SEARCH> cur{nb ? const_bounds(a.bounds + sp.bound_begin) : nullptr, nb, j0, 0, 0, JABAS_MAX_GROUPS, {}};
    // Eight fp32 workers with pair products, one tile in flight, take every tile by itself: the path over full tiles beside it costs 80
    // registers, for SGD (235 -> 154) and without an optimizer (230 -> 145) one wave per SIMD of three, for AdamW (250 -> 169) a third of the
    // spilled scalars. 3 M elements, both paths -> this: SGD 40.2 -> 35.0 us, AdamW 43.5 -> 41.2, no optimizer 30.2 -> 26.4; 12 M 122.5 -> 119.2,
    // 136.3 -> 133.5, 88.5 -> 83.6; 40 M SGD 369 -> 366, AdamW 426 -> 431. Not amsgrad: 3 M 47.5 -> 45.3, but 12 M 152.2 -> 155.3, 40 M 488 -> 499.
    constexpr bool ONE_BY_ONE = K <= 8 && U == 1 && OPT != OPT_AMS;
    for (uint32_t lt = lt0; lt < lt1;) {
        const uint64_t e0 = static_cast<uint64_t>(lt) * TE;
        uint32_t nfull = 0;
        // spans beyond 32-bit byte offsets go tile by tile
        if (!ONE_BY_ONE && e0 >= sp.lo && (!narrow_addressing(K, SL) || sp.narrow_ok)) {
            const uint64_t fit = (sp.hi - e0) / TE;
            const uint32_t left = lt1 - lt;
            nfull = fit < left ? static_cast<uint32_t>(fit) : left;
            // a workgroup's tiles are a chunk's or a part of them: one worker's statistics 60 M elements 36.0 -> 32.7 us (bf16), 46.5 ->
            // 45.9 (fp32); in other kernels the registers fall out worse (K = 4 SGD with replicas 212 -> 217, clipped Adam 1390 -> 1399)
            if constexpr (K == 1 && OPT == OPT_NONE && SL != 0) __builtin_assume(nfull <= CT);
        }
        if (nfull >= static_cast<uint32_t>(LEAST)) {
            lt += nfull - fast_run<K, DT, OPT, SL, HD, U, LEAST>(sp, e0, nfull, a, cur, clip, use_s1, load_s1, out, acc);
        } else {
            single_tile<K, DT, OPT, SL, HD>(sp, e0, a, cur, clip, use_s1, load_s1, out, acc);
            lt += 1;
        }
    }
}

// Statistics kernels carry two copies of the arithmetic: one with the default halves
// (even worker -> A, odd -> B) resolved at compile time, one driven by the half mask.
template <int K, int DT, int OPT, int SL, bool SEARCH, class A, class SP>
__device__ __forceinline__ void run_chunk(const SP& sp, uint32_t lt0, uint32_t lt1, uint32_t j0, const A& a,
                                          typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    if constexpr (SL) {
        constexpr uint32_t kDefaultMask = 0xAAAAu & ((1u << K) - 1u);
        if (a.half_mask == kDefaultMask) span_range<K, DT, OPT, SL, true, SEARCH>(sp, lt0, lt1, j0, a, acc);
        else span_range<K, DT, OPT, SL, false, SEARCH>(sp, lt0, lt1, j0, a, acc);
    } else {
        span_range<K, DT, OPT, 0, true, SEARCH>(sp, lt0, lt1, j0, a, acc);
    }
}

// Workgroup sum of NS per-thread accumulators -> one partial row, fp64 accumulators (fp32 gradients).
// Through LDS rather than wave shuffles: NS stores + 16 loads per thread instead of ~18 DPP-and-add
// instructions per value, which matters because a workgroup only covers a few thousand elements.
//   stage 1  thread (v, part) adds entries part, part+16, ..., part+240 of value v (in order);
//   stage 2  the 16 parts of a value sit in one 16-lane row: DPP row reduction.
// BS / 16 values go through the table at a time (16 with 256 threads), so rows wider than that take several
// passes over a table of 32 KB instead of one of up to 80 (pair products of eight workers: 40 values).
// The order is fixed, so the row is bit-identical from run to run.
template <int NS, int BS>
__device__ __forceinline__ void flush_stats(double (&acc)[NS], double* row) {
    constexpr int kParts = 16;                       // lanes of one DPP row
    constexpr int kPerPass = BS / kParts;            // values reduced per pass
    constexpr int kBuf = NS < kPerPass ? NS : kPerPass;
    __shared__ double buf[kBuf][BS];
    const int tid = threadIdx.x;
#pragma unroll
    for (int v0 = 0; v0 < NS; v0 += kPerPass) {
        if (v0) __syncthreads();                     // the table is read out before it is filled again
#pragma unroll
        for (int i = 0; i < kPerPass; ++i)
            if (v0 + i < NS) buf[i][tid] = acc[v0 + i];
        __syncthreads();
        if (tid < (NS - v0) * kParts) {              // at most kPerPass * 16 = BS threads
            const int v = tid >> 4, part = tid & 15;
            double s = buf[v][part];
#pragma unroll
            for (int i = 1; i < BS / kParts; ++i) s += buf[v][i * kParts + part];
            s += dpp_move<0xB1, 0xf>(s);     // quad_perm [1,0,3,2]
            s += dpp_move<0x4E, 0xf>(s);     // quad_perm [2,3,0,1]
            s += dpp_move<0x141, 0xf>(s);    // row_half_mirror
            s += dpp_move<0x140, 0xf>(s);    // row_mirror
            if (part == 0) row[v0 + v] = s;
        }
    }
}

template <int CTRL> __device__ __forceinline__ float dpp_move_f32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

// The same for fp32 accumulators (bf16 gradients). The sums of a 16-lane row are formed first, in fp32 by
// DPP (one instruction per step and value, no LDS traffic, no wait); only one entry per row and value goes
// through LDS, and what follows the barrier is short: thread (v, part) adds entries part, part+16, ... of
// value v in fp64 and the 16 parts meet by DPP. Every lane of the workgroup is active here.
template <int NS, int BS>
__device__ __forceinline__ void flush_stats(float (&acc)[NS], double* row) {
    constexpr int kParts = 16;
    constexpr int kRows = BS / 16;                   // 16-lane rows of the workgroup
    constexpr int kPerPass = BS / kParts;
    __shared__ float buf[NS][kRows];
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        float v = acc[i];
        v += dpp_move_f32<0xB1>(v);          // quad_perm [1,0,3,2]
        v += dpp_move_f32<0x4E>(v);          // quad_perm [2,3,0,1]
        v += dpp_move_f32<0x141>(v);         // row_half_mirror
        v += dpp_move_f32<0x140>(v);         // row_mirror
        if ((tid & 15) == 0) buf[i][tid >> 4] = v;
    }
    __syncthreads();
#pragma unroll
    for (int v0 = 0; v0 < NS; v0 += kPerPass) {
        if (tid < (NS - v0) * kParts) {
            const int v = v0 + (tid >> 4), part = tid & 15;
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < (kRows + kParts - 1) / kParts; ++i)
                if (i * kParts + part < kRows) s += static_cast<double>(buf[v][i * kParts + part]);
            s += dpp_move<0xB1, 0xf>(s);
            s += dpp_move<0x4E, 0xf>(s);
            s += dpp_move<0x141, 0xf>(s);
            s += dpp_move<0x140, 0xf>(s);
            if (part == 0) row[v] = s;
        }
    }
}

// The chunk of workgroup b: a names the launch (spans, chunk table), s the step's scalars (a itself, or the
// view of the device block).
template <int K, int DT, int OPT, int SL, class A>
__device__ __forceinline__ void workgroup_chunk(const KArgs& a, const A& s, uint32_t b,
                                                typename StatAcc<DT>::type (&acc)[NStats<K, SL>::value]) {
    constexpr int BS = launch_block(K, DT, OPT, SL);
    constexpr uint32_t CT = launch_chunk_tiles(K, DT, OPT, SL);     // the host cuts the chunk table for the same shape
    constexpr uint64_t TE = static_cast<uint64_t>(BS) * 4;
    const uint32_t per = CT >> a.split_log2;     // tiles of this workgroup
    if (a.use_inline) {
        const SpanDev& sp = a.span0;
        const uint32_t tiles = static_cast<uint32_t>((sp.hi + TE - 1) / TE);
        const uint32_t lt0 = b * per;
        const uint32_t lt1 = lt0 + per < tiles ? lt0 + per : tiles;
        run_chunk<K, DT, OPT, SL, true>(sp, lt0, lt1, 0, s, acc);
    } else {
        // The plan's tables are not written while a launch that names them runs: read through the constant
        // address space, their fields are loaded like kernel arguments (uniform loads the compiler may move,
        // repeat or keep as it likes) instead of being fetched again after every store that might alias them.
        typedef const __attribute__((address_space(4))) ChunkDesc* ConstChunk;
        typedef __attribute__((address_space(4))) SpanDev ConstSpan;
        ConstChunk cp = (ConstChunk)(a.chunks + (b >> a.split_log2));
        const uint32_t c_span = cp->span, c_bound0 = cp->bound0;
        const uint32_t lt0 = cp->tile0 + (b & ((1u << a.split_log2) - 1u)) * per;     // at or beyond the span's end: nothing to do
        const ConstSpan& sp = *(const ConstSpan*)(a.spans + c_span);
        const uint32_t tiles = static_cast<uint32_t>((sp.hi + TE - 1) / TE);
        const uint32_t lt1 = lt0 + per < tiles ? lt0 + per : tiles;
        run_chunk<K, DT, OPT, SL, false>(sp, lt0, lt1, c_bound0, s, acc);
    }
}

// DYN: the step's scalars are read from the device block a.dyn names (a launch that a HIP graph replays
// with another learning rate or Adam step) instead of from the kernel arguments.
template <int K, int DT, int OPT, int SL, bool DYN>
__global__ void __launch_bounds__(launch_block(K, DT, OPT, SL)) fused_kernel(const KArgs a) {
    constexpr int NS = NStats<K, SL>::value;
    constexpr int BS = launch_block(K, DT, OPT, SL);
    const uint32_t b = blockIdx.x;
    typename StatAcc<DT>::type acc[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) acc[i] = 0;
    if constexpr (DYN) {
        const DynView s(a);
        workgroup_chunk<K, DT, OPT, SL>(a, s, b, acc);
    } else {
        workgroup_chunk<K, DT, OPT, SL>(a, a, b, acc);
    }
    if constexpr (SL) flush_stats<NS, BS>(acc, a.partials + static_cast<uint64_t>(b) * NS);   // compact rows of 4 + K
}

template <int K, int DT, int OPT, int SL>
int launch_one(const KArgs& a, unsigned grid, hipStream_t stream, bool dyn) {
    // Residency cap through idle dynamic LDS (160 KB per CU). Fewer resident workgroups keep the
    // streamed window of every buffer more compact, which the memory system rewards on write-heavy
    // mixes as long as the kernel does not need the waves to hide its own arithmetic. Measured (A/B in
    // one process, and over whole bench runs with rotating buffers): Adam/AdamW at K <= 4 with fp32
    // gradients gains 0-4 % without statistics at 5 workgroups per CU instead of the 6 its registers
    // allow, and 0.2-2.4 % with statistics at 3 workgroups per CU instead of 4 (more with replica
    // weights to refresh); SGD kernels, bf16 gradients and K > 4 lose or stay flat.
#ifndef JABAS_IDLE_LDS_BYTES
#define JABAS_IDLE_LDS_BYTES 32768u
#endif
#ifndef JABAS_STATS_LDS_BYTES
#define JABAS_STATS_LDS_BYTES 53248u      // per workgroup, flush_stats' own table included: three workgroups per CU
#endif
    // An aggregate with statistics and no optimizer, K = 2..4 with fp32 gradients, where it reads 340 MB of them or more (their
    // registers allow seven or eight workgroups per CU): five where four workers' aggregate is written, six otherwise. Time against no
    // cap, aggregate in place, full rows / similarity sums: K = 4 five 25 M elements 0.984 / 0.973, 95 M 0.965 / 0.953; K = 3 six
    // 37 M 0.983 / 0.983, 119 M 0.970 / 0.972; K = 2 six 50 M 1.005 / 1.000, 158 M 0.974 / 0.961, read only 75 M 0.971 / 0.964; GNMT's
    // clipped step, whose first launch this is, 1413 -> 1383 us. Shorter launches wait for their last workgroups instead and lose:
    // 12 M elements K = 2 six 1.03 / 1.06, 9 M K = 3 five 1.06 / 1.08; and two workers' aggregate loses at five at any length (158 M 1.04).
#ifndef JABAS_AGG_LDS_BYTES
#define JABAS_AGG_LDS_BYTES 32768u
#endif
#ifndef JABAS_AGG_FEW_LDS_BYTES
#define JABAS_AGG_FEW_LDS_BYTES 26624u
#endif
#ifndef JABAS_AGG_CAP_FROM
#define JABAS_AGG_CAP_FROM 40960u         // gradient streams times workgroups of 2048 elements
#endif
    constexpr bool capped = OPT == OPT_ADAM && K <= 4 && DT == JABAS_F32, capped_agg = OPT == OPT_NONE && SL && K > 1 && K <= 4 && DT == JABAS_F32;
    constexpr unsigned flush_bytes = imin(NStats<K, SL>::value, launch_block(K, DT, OPT, SL) / 16) * launch_block(K, DT, OPT, SL) * 8u;   // flush_stats' fp64 table
    static_assert(!capped || !SL || flush_bytes < JABAS_STATS_LDS_BYTES, "the cap is what is left beside the table");
    const bool long_agg = capped_agg && static_cast<uint64_t>(grid) * K >= JABAS_AGG_CAP_FROM;
    const unsigned total = long_agg   ? (K > 3 && a.writes_agg ? JABAS_AGG_LDS_BYTES : JABAS_AGG_FEW_LDS_BYTES)
                         : !capped    ? 0u
                         : SL         ? JABAS_STATS_LDS_BYTES
                                      : JABAS_IDLE_LDS_BYTES;
    const unsigned table = SL ? flush_bytes : 0u, idle = total > table ? total - table : 0u;
    const dim3 block(launch_block(K, DT, OPT, SL));
    if constexpr (SL == JABAS_STATS_GRAM && K > JABAS_STATS_GRAM_MAX_K) {
        return static_cast<int>(hipErrorInvalidValue);              // refused by the front before it gets here
    } else {
        if constexpr (OPT == OPT_SGD || OPT == OPT_ADAM) {
            if (dyn) return static_cast<int>(launch_kernel(fused_kernel<K, DT, OPT, SL, true>, dim3(grid), block, idle, stream, a));
        } else {
            if (dyn) return static_cast<int>(hipErrorInvalidValue);     // refused by the front before it gets here
        }
        return static_cast<int>(launch_kernel(fused_kernel<K, DT, OPT, SL, false>, dim3(grid), block, idle, stream, a));
    }
}

}  // namespace

#define JABAS_CAT_(a, b) a##b
#define JABAS_CAT(a, b) JABAS_CAT_(a, b)

#define JABAS_DISPATCH(FN, ...)                                                              \
    const int key = (opt_class * 2 + (grad_dtype == JABAS_BF16 ? 1 : 0)) * 4 + stats;           \
    switch (key) {                                                                           \
        case 0: return FN<JABAS_K, JABAS_F32, OPT_NONE, 0>(__VA_ARGS__);                     \
        case 1: return FN<JABAS_K, JABAS_F32, OPT_NONE, 1>(__VA_ARGS__);                     \
        case 2: return FN<JABAS_K, JABAS_F32, OPT_NONE, 2>(__VA_ARGS__);                     \
        case 3: return FN<JABAS_K, JABAS_F32, OPT_NONE, 3>(__VA_ARGS__);                     \
        case 4: return FN<JABAS_K, JABAS_BF16, OPT_NONE, 0>(__VA_ARGS__);                    \
        case 5: return FN<JABAS_K, JABAS_BF16, OPT_NONE, 1>(__VA_ARGS__);                    \
        case 6: return FN<JABAS_K, JABAS_BF16, OPT_NONE, 2>(__VA_ARGS__);                    \
        case 7: return FN<JABAS_K, JABAS_BF16, OPT_NONE, 3>(__VA_ARGS__);                    \
        case 8: return FN<JABAS_K, JABAS_F32, OPT_SGD, 0>(__VA_ARGS__);                      \
        case 9: return FN<JABAS_K, JABAS_F32, OPT_SGD, 1>(__VA_ARGS__);                      \
        case 10: return FN<JABAS_K, JABAS_F32, OPT_SGD, 2>(__VA_ARGS__);                     \
        case 11: return FN<JABAS_K, JABAS_F32, OPT_SGD, 3>(__VA_ARGS__);                     \
        case 12: return FN<JABAS_K, JABAS_BF16, OPT_SGD, 0>(__VA_ARGS__);                    \
        case 13: return FN<JABAS_K, JABAS_BF16, OPT_SGD, 1>(__VA_ARGS__);                    \
        case 14: return FN<JABAS_K, JABAS_BF16, OPT_SGD, 2>(__VA_ARGS__);                    \
        case 15: return FN<JABAS_K, JABAS_BF16, OPT_SGD, 3>(__VA_ARGS__);                    \
        case 16: return FN<JABAS_K, JABAS_F32, OPT_ADAM, 0>(__VA_ARGS__);                    \
        case 17: return FN<JABAS_K, JABAS_F32, OPT_ADAM, 1>(__VA_ARGS__);                    \
        case 18: return FN<JABAS_K, JABAS_F32, OPT_ADAM, 2>(__VA_ARGS__);                    \
        case 19: return FN<JABAS_K, JABAS_F32, OPT_ADAM, 3>(__VA_ARGS__);                    \
        case 20: return FN<JABAS_K, JABAS_BF16, OPT_ADAM, 0>(__VA_ARGS__);                   \
        case 21: return FN<JABAS_K, JABAS_BF16, OPT_ADAM, 1>(__VA_ARGS__);                   \
        case 22: return FN<JABAS_K, JABAS_BF16, OPT_ADAM, 2>(__VA_ARGS__);                   \
        case 23: return FN<JABAS_K, JABAS_BF16, OPT_ADAM, 3>(__VA_ARGS__);                   \
        case 24: return FN<JABAS_K, JABAS_F32, OPT_AMS, 0>(__VA_ARGS__);                     \
        case 25: return FN<JABAS_K, JABAS_F32, OPT_AMS, 1>(__VA_ARGS__);                     \
        case 26: return FN<JABAS_K, JABAS_F32, OPT_AMS, 2>(__VA_ARGS__);                     \
        case 27: return FN<JABAS_K, JABAS_F32, OPT_AMS, 3>(__VA_ARGS__);                     \
        case 28: return FN<JABAS_K, JABAS_BF16, OPT_AMS, 0>(__VA_ARGS__);                    \
        case 29: return FN<JABAS_K, JABAS_BF16, OPT_AMS, 1>(__VA_ARGS__);                    \
        case 30: return FN<JABAS_K, JABAS_BF16, OPT_AMS, 2>(__VA_ARGS__);                    \
        case 31: return FN<JABAS_K, JABAS_BF16, OPT_AMS, 3>(__VA_ARGS__);                    \
        default: return -1;                                                                  \
    }

int JABAS_CAT(launch_fused_k, JABAS_K)(int grad_dtype, int opt_class, int stats, int dyn, const KArgs& a,
                                       unsigned grid, hipStream_t stream) {
    JABAS_DISPATCH(launch_one, a, grid, stream, dyn != 0)
}

}  // namespace jabas
