// K x K Gram matrix of the K worker gradients of one span: gram[a][b] = sum_e g_a[e]*g_b[e].
// Fixed order of operations: bit-identical run to run.
//   few workers    grid-stride over 4-element vectors, exact fp64 products of the fp32 (or widened bf16) values,
//                  K(K+1)/2 fp64 accumulators per thread on the vector ALU, summed over the wave on the fp64 matrix
//                  cores -> LDS -> one packed partial row per workgroup (K <= 5 for fp32 gradients, K <= 7 for bf16);
//   more, to 16    fp32 gradients: fp64 matrix cores, v_mfma_f64_4x4x4 over 4 x 4 blocks of worker pairs, fed
//                  from registers (gram_mfma_kernel below), still exact products and fp64 sums;
//                  bf16 gradients: bf16 matrix cores, exact fp32 products, fp32 running sums over short runs,
//                  then fp64 (gram_bf16_mfma_kernel).
// Then a finalize that sums the workgroup rows in a fixed order, four entries of the rows per workgroup.
#include "jabas_internal.h"

#ifndef JABAS_GRAM_VALU_MAX_K
#define JABAS_GRAM_VALU_MAX_K 5
#endif

#ifndef JABAS_GRAM_GRID
#define JABAS_GRAM_GRID 1024
#endif

namespace jabas {
namespace {

#ifndef JABAS_GRAM_VALU_MAX_K_BF16
#define JABAS_GRAM_VALU_MAX_K_BF16 7
#endif
// Up to here the vector-ALU kernel, beyond it the matrix cores. Both on fp32 gradients of 65 k / 300 k / 1.2 M / 25.6 M /
// 67 M / 100 M elements, whole call in us, vector ALU against matrix cores (1024 workgroups and an earlier finalize on both sides):
//   K = 4   5.9 / 7.1 /  9.3 /  68.5 / 165.5 / 244.3   against   5.9 / 8.1 / 10.2 /  69.7 / 180.6 / 260.9
//   K = 5   5.9 / 7.6 / 10.2 /  85.6 / 218.6 / 327.1   against   6.2 / 9.0 / 11.9 /  90.1 / 227.7 / 329.0
//   K = 6   6.1 / 9.6 / 13.4 / 101.1 / 260.1 / 395.5   against   6.3 / 9.2 / 12.2 / 102.5 / 261.0 / 381.8
//   K = 7   6.5 / 10.2 / 14.8 / 117.8 / 325.8 / 473.3  against   6.4 / 9.3 / 12.7 / 116.7 / 298.2 / 440.1
// The vector ALU also sums in chains a sixteenth as long: on 100 M elements the diagonal is 7e-16 off against 7e-15. bf16 gradients change
// at eight workers, where the matrix cores' sums are fp32 over short runs: up to seven every sum stays fp64.
constexpr int gram_valu_max_k(int grad_dtype) { return grad_dtype == JABAS_BF16 ? JABAS_GRAM_VALU_MAX_K_BF16 : JABAS_GRAM_VALU_MAX_K; }

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bits_to_float(uint32_t u) { return __builtin_bit_cast(float, u); }

template <int DT> struct GramLoad;
template <> struct GramLoad<JABAS_F32> {
    static constexpr int EPT = 4;
    using Raw = f32x4;
    static __device__ __forceinline__ Raw raw(const void* base, uint64_t e) {
        return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + e));
    }
    static __device__ __forceinline__ float elem(const Raw& r, int i) { return r[i]; }
    // elements of the vector at e that lie in [lo, hi), zeros for the others: nothing outside the span is read
    static __device__ __forceinline__ Raw edge(const void* base, uint64_t e, uint64_t lo, uint64_t hi) {
        Raw r;
#pragma unroll
        for (int i = 0; i < EPT; ++i) r[i] = (e + i >= lo && e + i < hi) ? static_cast<const float*>(base)[e + i] : 0.0f;
        return r;
    }
    static __device__ __forceinline__ void vec(const void* base, uint64_t e, float (&x)[4]) {
        const f32x4 r = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + e));
        x[0] = r.x; x[1] = r.y; x[2] = r.z; x[3] = r.w;
    }
    static __device__ __forceinline__ float one(const void* base, uint64_t e) { return static_cast<const float*>(base)[e]; }
};
template <> struct GramLoad<JABAS_BF16> {
    static constexpr int EPT = 4;
    static __device__ __forceinline__ void vec(const void* base, uint64_t e, float (&x)[4]) {
        const u32x2 r = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(base) + e));
        x[0] = bits_to_float(r.x << 16); x[1] = bits_to_float(r.x & 0xffff0000u);
        x[2] = bits_to_float(r.y << 16); x[3] = bits_to_float(r.y & 0xffff0000u);
    }
    static __device__ __forceinline__ float one(const void* base, uint64_t e) {
        return bits_to_float(static_cast<uint32_t>(static_cast<const uint16_t*>(base)[e]) << 16);
    }
};

// Running sums per product, and 1024 / sums workgroups: the vectors of a thread go to its sums in turn, so a sum is a chain of
// as many additions as with 1024 workgroups and one. Half the workgroups with one sum were 1.2 to 3.7 times as far from the
// exact sums from 12 M elements on.
constexpr int gram_valu_sums(int K, int grad_dtype) { return grad_dtype == JABAS_F32 && K >= 3 ? 2 : 1; }

template <int K, int DT>
__global__ void __launch_bounds__(kBlock) gram_kernel(const SpanDev sp, double* partials) {
    using L = GramLoad<DT>;
    constexpr int EPT = L::EPT, S = gram_valu_sums(K, DT);
    constexpr int NP = K * (K + 1) / 2;
    double acc[S][NP];
#pragma unroll
    for (int u = 0; u < S; ++u)
#pragma unroll
        for (int i = 0; i < NP; ++i) acc[u][i] = 0.0;

    const uint64_t nvec = (sp.hi + EPT - 1) / EPT;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    auto add = [&](uint64_t v, double (&sum)[NP]) {
        const uint64_t e = v * EPT;
        float g[K][EPT];
        if (e >= sp.lo && e + EPT <= sp.hi) {
#pragma unroll
            for (int k = 0; k < K; ++k) L::vec(sp.g[k], e, g[k]);
        } else {
#pragma unroll
            for (int i = 0; i < EPT; ++i) {
                const bool live = (e + i >= sp.lo) && (e + i < sp.hi);
#pragma unroll
                for (int k = 0; k < K; ++k) g[k][i] = live ? L::one(sp.g[k], e + i) : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            double d[K];
#pragma unroll
            for (int k = 0; k < K; ++k) d[k] = static_cast<double>(g[k][i]);
            int idx = 0;
#pragma unroll
            for (int a = 0; a < K; ++a)
#pragma unroll
                for (int b = 0; b <= a; ++b, ++idx) sum[idx] = __builtin_fma(d[a], d[b], sum[idx]);
        }
    };
    for (uint64_t v = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; v < nvec; v += S * stride) {
        add(v, acc[0]);
        if constexpr (S == 2) {
            if (v + stride < nvec) add(v + stride, acc[1]);
        }
    }
    if constexpr (S == 2) {
#pragma unroll
        for (int i = 0; i < NP; ++i) acc[0][i] += acc[1][i];
    }

    // Sum of every product over the wave's lanes on the fp64 matrix cores: lane j + 4 b + 16 i supplies entry (j, i) of
    // product b of v_mfma_f64_4x4x4 as the left operand and (i, j) as the right one. With ones on the other side the first
    // adds lanes 16 apart (entry (j, *) of its result is the sum over i), the second the four j: every lane then holds the
    // sum of the 16 lanes with its b, and lanes 0, 4, 8 and 12 write the four. Multiplying by one is exact, the sums are
    // fp64. Two instructions per product, where a tree of wave shuffles takes twelve LDS permutations: 1.2 M elements,
    // whole call, K = 5 fp32 22.0 -> 16.5 us, K = 7 bf16 34.8 -> 24.4 (9.4 and 11.4 with the finalize below and 512 workgroups for K = 5).
    __shared__ double red[kWaves][4][NP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const double q = __builtin_amdgcn_mfma_f64_4x4x4f64(acc[0][i], 1.0, 0.0, 0, 0, 0);
        const double v = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, q, 0.0, 0, 0, 0);
        if ((lane & 51) == 0) red[wave][lane >> 2][i] = v;
    }
    __syncthreads();
    if (threadIdx.x < NP) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            s += ((red[w][0][threadIdx.x] + red[w][1][threadIdx.x]) + red[w][2][threadIdx.x]) + red[w][3][threadIdx.x];
        partials[static_cast<uint64_t>(blockIdx.x) * JABAS_GRAM_STRIDE + threadIdx.x] = s;
    }
}

// Sums the workgroup rows and writes the symmetric matrix, four neighbouring entries of the rows per workgroup: lane =
// entry + 4 * row, so a wave's load covers 32 contiguous bytes of sixteen rows, every thread has four loads in flight (1024
// rows: all of them) and a wider row only adds workgroups. Thread (entry, class) adds rows class, class + 256, ... in order;
// the 256 sums of an entry meet by row rotations, one LDS table and a second round of the same: the order depends on the
// number of rows alone, the result not on timing.
// BLOCKS: rows of the matrix-core kernels, entry [p][4 i + j] is the product of workers 4 ga + i and 4 gb + j of pair
// p = (ga <= gb); otherwise packed rows, entry a (a + 1) / 2 + b of workers b <= a.
// Bound by its launch and one trip to memory. One workgroup for all entries (packed rows), and two launches, a fold to 32
// rows and one workgroup (blocks), cost more; whole calls on 0.3 / 0.7 / 1.2 / 25.6 M elements, us, before -> now:
//   fp32 K = 2   7.9 / 7.9 / 8.9 / 36.1  ->  7.6 / 7.5 / 7.5 / 34.9       fp32 K = 8    10.0 / 11.6 / 13.6 / 122.8  ->  8.8 / 10.2 / 12.4 / 122.6
//   fp32 K = 5   8.8 / 10.7 / 11.1 / 85.6  ->  8.2 / 8.9 / 10.3 / 84.4     fp32 K = 16   13.7 / 17.4 / 22.6 / 257.3  ->  12.1 / 15.9 / 21.7 / 257.7
//   bf16 K = 7   11.4 / 11.9 / 13.7 / 65.6  ->  9.4 / 9.5 / 11.1 / 63.0    bf16 K = 16   14.8 / 18.8 / 22.3 / 133.6  ->  12.9 / 17.1 / 21.4 / 132.8
constexpr int kGramFinalizeBlock = 1024, kGramFinalizeSlots = 4;
constexpr unsigned kGramFinalizeClasses = kGramFinalizeBlock / kGramFinalizeSlots;
template <bool BLOCKS>
__global__ void __launch_bounds__(kGramFinalizeBlock) gram_finalize_kernel(int K, const double* partials, unsigned grid,
                                                                         double* gram_out) {
    __shared__ double table[kGramFinalizeBlock / 16][kGramFinalizeSlots];
    const int G = (K + 3) / 4;
    const int width = BLOCKS ? G * (G + 1) / 2 * 16 : K * (K + 1) / 2;
    const int t = threadIdx.x, entry = static_cast<int>(blockIdx.x) * kGramFinalizeSlots + (t & (kGramFinalizeSlots - 1));
    const double* col = partials + (entry < width ? entry : width - 1);
    double s = 0.0;
    for (unsigned r = t / kGramFinalizeSlots; r < grid; r += 4 * kGramFinalizeClasses) {
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {            // a row beyond the last repeats the last and is dropped
            const unsigned c = r + i * kGramFinalizeClasses;
            v[i] = col[static_cast<uint64_t>(c < grid ? c : grid - 1) * JABAS_GRAM_STRIDE];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s += r + i * kGramFinalizeClasses < grid ? v[i] : 0.0;
    }
    s += dpp_move<0x128, 0xf>(s);                // row_ror:8, row_ror:4: the four classes of a 16-lane row, per entry
    s += dpp_move<0x124, 0xf>(s);
    if ((t & 15) < kGramFinalizeSlots) table[t >> 4][t & 15] = s;
    __syncthreads();
    if (t < 64) {                                // one wave: 64 sums of an entry, four per lane, then over the lanes
        const int c = t >> 2, v = t & (kGramFinalizeSlots - 1);
        double sum = ((table[c][v] + table[16 + c][v]) + table[32 + c][v]) + table[48 + c][v];
        sum += dpp_move<0x128, 0xf>(sum);
        sum += dpp_move<0x124, 0xf>(sum);
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        int lo = 0, hi = 0;
        if constexpr (BLOCKS) {                  // the workgroup holds row i of pair p: p, then ga, from its index
            int p = static_cast<int>(blockIdx.x) >> 2, ga = 0;
            while (p >= G - ga) p -= G - ga++;
            lo = 4 * ga + (static_cast<int>(blockIdx.x) & 3);
            hi = 4 * (ga + p) + v;
        } else {
            while ((hi + 1) * (hi + 2) / 2 <= entry) ++hi;
            lo = entry - hi * (hi + 1) / 2;
        }
        if (t < kGramFinalizeSlots && lo <= hi && hi < K) {      // one triangle, mirrored: symmetric bit for bit
            gram_out[lo * JABAS_GRAM_MAX_K + hi] = sum;
            gram_out[hi * JABAS_GRAM_MAX_K + lo] = sum;
        }
    } else if (blockIdx.x == 0 && t - 64 < JABAS_GRAM_STRIDE) {
        const int o = t - 64;
        if (o / JABAS_GRAM_MAX_K >= K || o % JABAS_GRAM_MAX_K >= K) gram_out[o] = 0.0;
    }
}
static_assert(kGramFinalizeBlock >= 64 + JABAS_GRAM_STRIDE, "one thread per entry of the matrix beside the summing wave");


// ---- K >= 6: fp64 matrix cores, 4 x 4 blocks ----------------------------------------------------------
// The Gram matrix is a contraction over the elements, X X^T with X the K x N matrix of the workers'
// gradients. The workers are cut into G = ceil(K / 4) groups of four; v_mfma_f64_4x4x4 (four independent
// 4 x 4 x 4 products per instruction) forms, for one pair of groups (ga <= gb), the 4 x 4 block of products
// over four elements in each of its four products. Lane l is
// worker l % 4 of every group and vector l / 4 of a 64-element block: it loads ONE 16-byte vector per group
// (a wave reads 256 contiguous bytes of each worker) and feeds round r of every pair from registers,
// A = element r of its vector of group ga, B = element r of its vector of group gb: no LDS, no shuffles,
// G(G+1)/2 running sums per lane instead of K(K+1)/2 register pairs per thread (which is what limits the
// vector-ALU form to few workers). Products of widened fp32 values are exact in fp64 and the order is fixed.
// Per 64 elements: 4 G(G+1)/2 MFMAs and 4 G conversions per wave, against 36 fp64 multiply-adds and 8
// conversions PER ELEMENT AND THREAD at K = 8 on the vector ALU.
#ifndef JABAS_GRAM_RUN_F32
#define JABAS_GRAM_RUN_F32 2
#endif
// 64-element blocks in a run of a wave
constexpr int kGramRunBlocks = JABAS_GRAM_RUN_F32;
constexpr uint64_t kGramShortF32 = 1u << 21;           // fewer elements: half the workgroups (gram_grid)

// S: running sums per pair of groups; a wave's runs go to them in turn. Two with half the workgroups (gram_grid): as many runs per
// sum as with all of them and one, which half the workgroups and one sum were 1.2 to 2.3 times as far from the exact sums as.
template <int G, int S>
__global__ void __launch_bounds__(kBlock) gram_mfma_kernel(const SpanDev sp, int K, double* partials) {
    using L = GramLoad<JABAS_F32>;
    constexpr int P = G * (G + 1) / 2;
    constexpr uint64_t kRun = static_cast<uint64_t>(kGramRunBlocks) * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = lane & 3;                           // worker inside its group
    const uint32_t lane_off = static_cast<uint32_t>(lane >> 2) * 4u;
    const void* base[G];
    bool live[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        live[g] = g * 4 + wi < K;
        base[g] = sp.g[live[g] ? g * 4 + wi : 0];
    }
    double acc[S][P];
#pragma unroll
    for (int u = 0; u < S; ++u)
#pragma unroll
        for (int p = 0; p < P; ++p) acc[u][p] = 0.0;
    // Runs that lie wholly in the span are [first, last); at most two others hold its ends.
    const uint64_t n_runs = (sp.hi + kRun - 1) / kRun, first = (sp.lo + kRun - 1) / kRun;
    const uint64_t last = sp.hi / kRun > first ? sp.hi / kRun : first;
    const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * kWaves;
    auto load = [&](uint64_t run, L::Raw (&x)[kGramRunBlocks][G]) {
#pragma unroll
        for (int u = 0; u < kGramRunBlocks; ++u)
#pragma unroll
            // a lane beyond the last worker reads worker 0's vector (the same line another lane of the
            // wave reads anyway) and drops it when it multiplies: no load waits for another
            for (int g = 0; g < G; ++g) x[u][g] = L::raw(base[g], run * kRun + u * 64 + lane_off);
    };
    auto multiply = [&](const L::Raw (&x)[kGramRunBlocks][G], double (&sum)[P]) {
#pragma unroll
        for (int u = 0; u < kGramRunBlocks; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double d[G];
#pragma unroll
                for (int g = 0; g < G; ++g) d[g] = live[g] ? static_cast<double>(L::elem(x[u][g], r)) : 0.0;
                int p = 0;
#pragma unroll
                for (int ga = 0; ga < G; ++ga)
#pragma unroll
                    for (int gb = ga; gb < G; ++gb, ++p)
                        sum[p] = __builtin_amdgcn_mfma_f64_4x4x4f64(d[ga], d[gb], sum[p], 0, 0, 0);
            }
    };
    // Bound by HBM reads. Two runs in flight per wave, the next one's loads issued before this one is multiplied; only whole
    // runs, so that the loop has no edge path. Whole call, one run in flight -> two, 25.6 M elements: K = 6 106.0 -> 102.5
    // us, K = 8 135.2 -> 124.5 (6.57 TB/s), K = 12 197.5 -> 189.0 (6.49), K = 13 226.8 -> 220.5, K = 16 259.1 -> 256.8;
    // 100 M: K = 8 502 -> 490, K = 12 743 -> 732, K = 16 991 -> 990. Over 240 random sizes from 65 k to 100 M: K = 6..8
    // 1.00-1.08 times as fast by decade half, K = 9..12 0.99-1.05 (0.99 around 600 k), K = 13..16 1.00-1.05. Runs half as
    // long or twice as long lose 2-5 %.
    const uint64_t id = static_cast<uint64_t>(blockIdx.x) * kWaves + wave;
    L::Raw x[kGramRunBlocks][G], y[kGramRunBlocks][G];
    uint64_t run = first + id;
    if (run < last) {
        load(run, x);
        while (true) {
            const bool more = (run += n_waves) < last;
            if (more) load(run, y);
            multiply(x, acc[0]);
            if (!more) break;
            const bool again = (run += n_waves) < last;
            if (again) load(run, x);
            multiply(y, acc[S - 1]);
            if (!again) break;
        }
    }
    // The ends go to the last waves, which have a run less when the runs do not come out even.
    const uint64_t n_ends = first + (n_runs > last ? n_runs - last : 0);
    for (uint64_t r = n_waves - 1 - id; r < n_ends; r += n_waves) {
        const uint64_t e0 = (r < first ? r : last + (r - first)) * kRun + lane_off;
#pragma unroll
        for (int u = 0; u < kGramRunBlocks; ++u) {
            const uint64_t e = e0 + u * 64;
            const bool whole = e >= sp.lo && e + L::EPT <= sp.hi;
#pragma unroll
            for (int g = 0; g < G; ++g) x[u][g] = whole ? L::raw(base[g], e) : L::edge(base[g], e, sp.lo, sp.hi);
        }
        multiply(x, acc[0]);
    }
    // The instruction's contraction index is lane / 16 and its four independent products are indexed by
    // (lane / 4) % 4; entry (i, j) of product b sits in lane j + 4 b + 16 i. Which of a lane's elements meets
    // which is therefore fixed by the lanes alone (A and B come from the same lane), and the four products
    // are partial sums over different elements of the same 4 x 4 block. Row of the workgroup: entry
    // [p][4 i + j] is the sum over the four products and the four waves (in that order) for pair p.
    __shared__ double red[kWaves][P][64];
#pragma unroll
    for (int p = 0; p < P; ++p) red[wave][p][lane] = S == 2 ? acc[0][p] + acc[S - 1][p] : acc[0][p];
    __syncthreads();
    for (int t = threadIdx.x; t < P * 16; t += kBlock) {
        const int p = t >> 4, i = (t >> 2) & 3, j = t & 3;
        const int l0 = j + 16 * i;
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s += ((red[w][p][l0] + red[w][p][l0 + 4]) + red[w][p][l0 + 8]) + red[w][p][l0 + 12];
        partials[static_cast<uint64_t>(blockIdx.x) * JABAS_GRAM_STRIDE + t] = s;
    }
}

// ---- bf16 gradients: bf16 matrix cores ------------------------------------------------------------------
// v_mfma_f32_4x4x4_16b_bf16 multiplies, in each of its 16 independent products, a 4 x 4 operand by a 4 x 4
// operand whose contraction index runs over the four bf16 values ONE lane supplies in a register pair. With the lane
// layout above (lane l = worker l % 4 of its group, vector l / 4 of the block) the raw loaded registers ARE
// the operands: no widening, no conversion, one instruction per pair of groups and four elements of every
// lane. A lane loads 16 bytes (two operands) per group; a wave reads 256 contiguous bytes of each worker.
// Products of bf16 values are exact in fp32; the instruction adds four of them to an fp32 running sum, which
// is moved into fp64 sums (LDS, per wave) after at most kGramBf16FlushRuns runs. A sum then holds at most 4 * 2 * (U / S) *
// kGramBf16FlushRuns products (U blocks of a run go to S sums; two vectors of four per block) and, in the first of them, those of
// the span's ends: 1024 to 2048, 4096 in the shape of four groups and very long spans. fp32 rounding stays near 1e-6 of
// |g_a| |g_b|, the order is fixed.
// Lanes beyond the last worker multiply worker 0's values into entries the finalize never reads.
template <int CTRL> __device__ __forceinline__ float gram_dpp_f32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(8))) u32x4_a8;     // element 0 of a bf16 buffer is 8-byte aligned, not more

constexpr int kGramBf16FlushRuns = 128;

// U: 128-element blocks in a run of a wave. S: running sums per pair of groups, which the blocks take in turn. EDGES: the
// loop takes the runs across the span's ends as well; otherwise it holds whole runs and the ends follow it, which keeps the
// conditional loads of single elements (U * G * 8 of them) out of its code: a cold launch fetches that code from memory.
template <int G, int U, int S, bool EDGES>
__global__ void __launch_bounds__(kBlock) gram_bf16_mfma_kernel(const SpanDev sp, int K, double* partials) {
    constexpr int P = G * (G + 1) / 2;
    constexpr uint64_t kRun = static_cast<uint64_t>(U) * 128;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = lane & 3;
    const uint32_t lane_off = static_cast<uint32_t>(lane >> 2) * 8u;
    const uint16_t* base[G];
#pragma unroll
    for (int g = 0; g < G; ++g) base[g] = static_cast<const uint16_t*>(sp.g[g * 4 + wi < K ? g * 4 + wi : 0]);
    // fp64 sums of the wave: [pair * 4 + i][16-lane row * 4 + j]
    __shared__ double sums[kWaves][P * 4][16];
    double* const wave_sums = &sums[0][0][0] + static_cast<size_t>(wave) * (P * 64);     // this wave's P * 64 sums, flat
    for (int i = lane; i < P * 64; i += 64) wave_sums[i] = 0.0;
    // the zeros are written by other lanes than the ones that add to them later: order the two within the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    f32x4 acc[S][P];
#pragma unroll
    for (int u = 0; u < S; ++u)
#pragma unroll
        for (int p = 0; p < P; ++p) acc[u][p] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // entry (i, j) of a product sits in register i of lane j + 4 * product: a rotation by 4 and by 8 inside the
    // 16-lane row adds the row's four products; lanes 0..3 of every row then own one fp64 sum each per register
    const bool owner = ((lane >> 2) & 3) == 0;
    const int col = (lane >> 4) * 4 + wi;
    auto flush = [&]() {
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                double sum = 0.0;
#pragma unroll
                for (int u = 0; u < S; ++u) {
                    float v = acc[u][p][i];
                    v += gram_dpp_f32<0x124>(v);    // row_ror:4
                    v += gram_dpp_f32<0x128>(v);    // row_ror:8
                    sum += static_cast<double>(v);
                }
                if (owner) sums[wave][p * 4 + i][col] += sum;
#pragma unroll
                for (int u = 0; u < S; ++u) acc[u][p][i] = 0.0f;
            }
    };
    auto load_edge = [&](uint64_t e, u32x4 (&v)[G]) {        // zeros for the elements beyond the span's ends, which are not read
        const bool whole = e >= sp.lo && e + 8 <= sp.hi;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (whole) {
                v[g] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a8*>(base[g] + e));
            } else {
                uint32_t h[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) h[i] = (e + i >= sp.lo && e + i < sp.hi) ? base[g][e + i] : 0u;
                v[g] = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
            }
        }
    };
    auto load = [&](uint64_t run, u32x4 (&x)[U][G]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t e = run * kRun + u * 128 + lane_off;
            if constexpr (EDGES) {
                load_edge(e, x[u]);
            } else {
#pragma unroll
                for (int g = 0; g < G; ++g) x[u][g] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a8*>(base[g] + e));
            }
        }
    };
    auto multiply_block = [&](const u32x4 (&v)[G], f32x4 (&sum)[P]) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            s16x4 d[G];
#pragma unroll
            for (int g = 0; g < G; ++g)
                d[g] = __builtin_bit_cast(s16x4, half ? u32x2{v[g].z, v[g].w} : u32x2{v[g].x, v[g].y});
            int p = 0;
#pragma unroll
            for (int ga = 0; ga < G; ++ga)
#pragma unroll
                for (int gb = ga; gb < G; ++gb, ++p) sum[p] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(d[ga], d[gb], sum[p], 0, 0, 0);
        }
    };
    auto multiply = [&](const u32x4 (&x)[U][G]) {
#pragma unroll
        for (int u = 0; u < U; ++u) multiply_block(x[u], acc[u % S]);
    };
    // The loop's runs are [first, last); at most two others hold the span's ends, taken block by block after it.
    const uint64_t n_runs = (sp.hi + kRun - 1) / kRun, first = EDGES ? 0 : (sp.lo + kRun - 1) / kRun;
    const uint64_t last = EDGES ? n_runs : sp.hi / kRun > first ? sp.hi / kRun : first;
    const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * kWaves;
    const uint64_t id = static_cast<uint64_t>(blockIdx.x) * kWaves + wave;
    const uint64_t n_ends = first + (n_runs > last ? n_runs - last : 0);
    auto ends = [&]() {                              // to the last waves, which have a run less when the runs do not come out even
        for (uint64_t r = n_waves - 1 - id; r < n_ends; r += n_waves) {
            const uint64_t e0 = (r < first ? r : last + (r - first)) * kRun + lane_off;
#pragma unroll 1
            for (int u = 0; u < U; ++u) {
                u32x4 v[G];
                load_edge(e0 + static_cast<uint64_t>(u) * 128, v);
                multiply_block(v, acc[0]);
            }
        }
    };
    // Bound by HBM reads from about 5 M elements on, below by the trips to memory and the epilogue.
    u32x4 x[U][G];
    uint64_t run = first + id;
    do {
        for (int n = 0; run < last && n < kGramBf16FlushRuns; ++n, run += n_waves) {
            load(run, x);
            multiply(x);
        }
        if constexpr (!EDGES) {
            if (run >= last) ends();
        }
        flush();                                     // the one copy of it: the code of a cold launch is fetched too
    } while (run < last);
    __syncthreads();
    // row of the workgroup, the format of gram_mfma_kernel: entry [p][4 i + j], rows then waves in order
    for (int t = threadIdx.x; t < P * 16; t += kBlock) {
        const int p = t >> 4, i = (t >> 2) & 3, j = t & 3;
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            s += ((sums[w][p * 4 + i][j] + sums[w][p * 4 + i][4 + j]) + sums[w][p * 4 + i][8 + j]) + sums[w][p * 4 + i][12 + j];
        partials[static_cast<uint64_t>(blockIdx.x) * JABAS_GRAM_STRIDE + t] = s;
    }
}

static_assert(JABAS_GRAM_VALU_MAX_K >= 4 && JABAS_GRAM_VALU_MAX_K_BF16 >= 4, "the matrix-core kernels start at two groups");
// Shapes of the bf16 matrix-core kernels. Whole calls in us, K = 8 / 12 / 16, before (one sum, ends in the loop, 1024
// workgroups, runs of 2 / 2 / 4 blocks) -> now:
//   0.3 M  8.8 / 10.5 / 12.9 -> 8.3 / 10.4 / 13.3      5 M   20.7 / 28.9 / 39.4 -> 19.1 / 27.1 / 35.4
//   1.2 M  9.9 / 13.9 / 21.4 -> 9.9 / 13.5 / 16.3      25 M  69.1 / 97.5 / 132.8 -> 65.4 / 95.0 / 128.0
//   four groups            two waves per SIMD fit, so 512 workgroups are resident: 1024 run in two rounds. Two sums per pair
//                          keep the fp32 chains as short as they were.
//   up to three groups     from kGramLongBf16 elements on the same with runs of four blocks; below, two blocks and one sum,
//                          1024 workgroups: longer runs leave waves idle (0.3 M, K = 8: 9.2), and two sums of two products
//                          each are 6 % further from the 64-bit result there than one of four.
//   four groups, very long from kGramVeryLongBf16 on the loop with the ends in it and 1024 workgroups, two resident per CU by
//                          idle LDS: 100 M elements of thirteen / fourteen / sixteen workers 405 / 431 / 478 us against
//                          408 / 438 / 488 with the shape above, three resident 438 / 451 / 494; 40 M 174 / 183 / 200 against
//                          165 / 177 / 197, 66 M 274 / 291 / 319 against 268 / 289 / 321.
#ifndef JABAS_GRAM_LONG_BF16
#define JABAS_GRAM_LONG_BF16 (1u << 21)
#endif
#ifndef JABAS_GRAM_VERY_LONG_BF16
#define JABAS_GRAM_VERY_LONG_BF16 (1u << 26)
#endif
constexpr uint64_t kGramLongBf16 = JABAS_GRAM_LONG_BF16, kGramVeryLongBf16 = JABAS_GRAM_VERY_LONG_BF16;

template <int G, int U, int S, bool EDGES>
int launch_gram_bf16_shape(int K, const SpanDev& sp, double* partials, unsigned grid, hipStream_t stream) {
    constexpr unsigned idle = EDGES ? 36 * 1024 : 0;     // beside the 20 KB of sums: two workgroups per CU of 160 KB
    return static_cast<int>(launch_kernel(gram_bf16_mfma_kernel<G, U, S, EDGES>, dim3(grid), dim3(kBlock), idle, stream, sp, K, partials));
}

int launch_gram_bf16_mfma(int K, const SpanDev& sp, double* partials, unsigned grid, hipStream_t stream) {
    const bool long_span = sp.hi >= kGramLongBf16;
    switch ((K + 3) / 4) {
        case 2: return long_span ? launch_gram_bf16_shape<2, 4, 2, false>(K, sp, partials, grid, stream)
                                 : launch_gram_bf16_shape<2, 2, 1, false>(K, sp, partials, grid, stream);
        case 3: return long_span ? launch_gram_bf16_shape<3, 4, 2, false>(K, sp, partials, grid, stream)
                                 : launch_gram_bf16_shape<3, 2, 1, false>(K, sp, partials, grid, stream);
        case 4: return sp.hi >= kGramVeryLongBf16 ? launch_gram_bf16_shape<4, 4, 1, true>(K, sp, partials, grid, stream)
                       : long_span                ? launch_gram_bf16_shape<4, 4, 2, false>(K, sp, partials, grid, stream)
                                                  : launch_gram_bf16_shape<4, 2, 2, false>(K, sp, partials, grid, stream);
        default: return -1;
    }
}

template <int K>
int launch_gram_k(int grad_dtype, const SpanDev& sp, double* partials, unsigned grid, hipStream_t stream) {
    if (grad_dtype == JABAS_BF16)
        return static_cast<int>(launch_kernel(gram_kernel<K, JABAS_BF16>, dim3(grid), dim3(kBlock), 0, stream, sp, partials));
    if constexpr (K <= JABAS_GRAM_VALU_MAX_K)
        return static_cast<int>(launch_kernel(gram_kernel<K, JABAS_F32>, dim3(grid), dim3(kBlock), 0, stream, sp, partials));
    return -1;
}

template <int S>
int launch_gram_mfma(int K, const SpanDev& sp, double* partials, unsigned grid, hipStream_t stream) {
    switch ((K + 3) / 4) {
        case 2: return static_cast<int>(launch_kernel(gram_mfma_kernel<2, S>, dim3(grid), dim3(kBlock), 0, stream, sp, K, partials));
        case 3: return static_cast<int>(launch_kernel(gram_mfma_kernel<3, S>, dim3(grid), dim3(kBlock), 0, stream, sp, K, partials));
        case 4: return static_cast<int>(launch_kernel(gram_mfma_kernel<4, S>, dim3(grid), dim3(kBlock), 0, stream, sp, K, partials));
        default: return -1;
    }
}

}  // namespace

// Most workgroups of a launch; hi: end of the span's element grid. 1024 unless half of them are faster:
//   bf16 matrix cores      with the shapes above
//   fp32 vector ALU        three to five workers, two sums each: K = 5, 25 M / 100 M elements 84.3 / 322 -> 80.3 / 304 us, K = 4
//                          65.5 / 243 -> 65.5 / 239, K = 3 equal, all equal below 2 M (K = 1 and 2 lose 10-50 %, bf16 up to 30 %)
//   fp32 matrix cores      short spans, whose waves have two or three runs each, two sums each: K = 9 / 13 / 16, 1.2 M elements
//                          15.5 / 20.4 / 21.7 -> 14.3 / 19.4 / 20.9 us, equal from 2.5 to 10 M; 25 M K = 8 122 -> 124, K = 9 151 -> 154
// Distance of the diagonal from the exact sums, 1024 workgroups / half of them with one sum / with two (mean over seeds):
//   K = 5   12 M 1.8 / 2.2 / 1.2e-16   25.6 M 2.6 / 5.9 / 2.1e-16   100 M 6.9 / 10.6 / 7.2e-16
//   K = 9   0.7 M 2.0 / 2.5 / 1.5e-16   1.2 M 3.1 / 4.6 / 2.2e-16   2.0 M 3.5 / 7.6 / 3.1e-16
unsigned gram_grid(int K, int grad_dtype, uint64_t hi) {
    const int groups = (K + 3) / 4;
    bool half;
    if (K <= gram_valu_max_k(grad_dtype)) half = gram_valu_sums(K, grad_dtype) == 2;
    else if (grad_dtype == JABAS_F32) half = hi < kGramShortF32;
    else half = groups == 4 ? hi < kGramVeryLongBf16 : hi >= kGramLongBf16;
    return half ? JABAS_GRAM_GRID / 2 : JABAS_GRAM_GRID;
}

int launch_gram(int K, int grad_dtype, const SpanDev& sp, double* partials, unsigned grid, hipStream_t stream) {
    if (K > gram_valu_max_k(grad_dtype))
        return grad_dtype == JABAS_BF16 ? launch_gram_bf16_mfma(K, sp, partials, grid, stream)
               : sp.hi < kGramShortF32      ? launch_gram_mfma<2>(K, sp, partials, grid, stream)
                                          : launch_gram_mfma<1>(K, sp, partials, grid, stream);
    switch (K) {
        case 1: return launch_gram_k<1>(grad_dtype, sp, partials, grid, stream);
        case 2: return launch_gram_k<2>(grad_dtype, sp, partials, grid, stream);
        case 3: return launch_gram_k<3>(grad_dtype, sp, partials, grid, stream);
        case 4: return launch_gram_k<4>(grad_dtype, sp, partials, grid, stream);
        case 5: return launch_gram_k<5>(grad_dtype, sp, partials, grid, stream);
        case 6: return launch_gram_k<6>(grad_dtype, sp, partials, grid, stream);
        case 7: return launch_gram_k<7>(grad_dtype, sp, partials, grid, stream);
        default: return -1;
    }
}

int launch_gram_finalize(int K, int grad_dtype, const double* partials, unsigned grid, double* gram_out, hipStream_t stream) {
    const unsigned G = (K + 3) / 4;
    const dim3 block(kGramFinalizeBlock);
    if (K > gram_valu_max_k(grad_dtype))
        return static_cast<int>(launch_kernel(gram_finalize_kernel<true>, dim3(G * (G + 1) / 2 * 16 / kGramFinalizeSlots), block, 0,
                                              stream, K, partials, grid, gram_out));
    return static_cast<int>(launch_kernel(gram_finalize_kernel<false>, dim3((K * (K + 1) / 2 + kGramFinalizeSlots - 1) / kGramFinalizeSlots),
                                          block, 0, stream, K, partials, grid, gram_out));
}

}  // namespace jabas
