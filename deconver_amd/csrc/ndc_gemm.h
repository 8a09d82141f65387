// The remaining GEMMs of the 1x1 projections on channel-first tensors, float32 and bf16:
//
//   tile_kernel    y[b] = epilogue(W x[b])        (forward and input gradient, layers/linear.py:53-58
//   parts_kernel                                   of the reference with its callers' tails; bf16 and float32)
//   sliced_kernel  the same over small grids
//   wgrad_kernel   gw = sum_b gz[b] x[b]^T,       (weight gradient, with the bias gradient
//                  gb = row sums of gz             sum_{b,v} gz from the same pass)
//
// What the streaming GEMM of ndc_pwgemm.h does not take ends up here: float32 storage, the wide
// levels whose weights do not fit LDS, odd voxel counts, small grids.  They are ordinary
// LDS-tiled matrix-instruction GEMMs; what is particular to them:
//
//   * Unit of staging is a 16-byte granule: 8 bf16 or 4 float32 values of consecutive k for one
//     row (one column) of the operand, which is what a lane hands v_mfma_f32_32x32x16_bf16, or,
//     element after element, four v_mfma_f32_32x32x2_f32.  A stage is 8 granules deep (64 bf16 or
//     32 float32 k-values); granule (row r, depth q) sits at slot q * rows + (r ^ q), so that
//     neither its writer (8 lanes along q, for operands contiguous in k) nor its readers (32 lanes
//     along r) meet a bank twice.
//   * float32 products are made of bf16 parts (see below) where matrix instructions are what a tile waits for.
//   * Whatever order the instruction takes its k-values in, both operands are filled by one rule
//     (lane half kb, element e <-> k = (2 step + kb) * E + e), so the products pair up.
//   * The weight comes in as it lies (float32, rows of W or of its transpose): no packing launch
//     and no cast copy.
//   * Voxel counts of any size and tensors of any alignment: ragged ends are filled with zeros
//     element by element, rows that are not 16-byte aligned are read with unaligned vector loads.
//
// Sums are float32 in a fixed order (partial results of the split voxel axis are added in order
// by a second launch): results are reproducible.  Device code only.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "ndc_common.h"
#include "ndc_epilogue.h"

#define NDC_INLINE __attribute__((always_inline))

namespace ndc {
namespace gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// the same at any element alignment
typedef u32x4 u32x4_a2 __attribute__((aligned(2), may_alias));
typedef u32x2 u32x2_a2 __attribute__((aligned(2), may_alias));

static const int kDepth = 8;              // granules per stage along k

template <typename T> struct Gran;        // E elements of consecutive k in 16 bytes
template <> struct Gran<float> {
    static constexpr int E = 4;
    static __device__ u32x4 pack(const float (&v)[4])
    {
        u32x4 r = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
        return r;
    }
    static __device__ float sum(u32x4 g)
    {
        return (__uint_as_float(g[0]) + __uint_as_float(g[1])) + (__uint_as_float(g[2]) + __uint_as_float(g[3]));
    }
    static __device__ f32x4 mma(u32x4 a, u32x4 b, f32x4 acc)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[j]), __uint_as_float(b[j]), acc, 0, 0, 0);
        return acc;
    }
    static __device__ f32x16 mma(u32x4 a, u32x4 b, f32x16 acc)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[j]), __uint_as_float(b[j]), acc, 0, 0, 0);
        return acc;
    }
};
template <> struct Gran<bf16_t> {
    static constexpr int E = 8;
    static __device__ u32x4 pack(const float (&v)[8])
    {
        u32x4 r = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
        return r;
    }
    static __device__ float sum(u32x4 g)
    {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s += __uint_as_float(g[i] << 16) + __uint_as_float(g[i] & 0xffff0000u);
        return s;
    }
    static __device__ f32x4 mma(u32x4 a, u32x4 b, f32x4 acc)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
    }
    static __device__ f32x16 mma(u32x4 a, u32x4 b, f32x16 acc)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
    }
};

// Granule slot.  Rows of a stage: a multiple of 32.
__device__ inline int slot(int rows, int q, int r) { return q * rows + (r ^ q); }

// E elements from `p` of which the first `have` exist (the rest read as zero)
template <typename T> __device__ inline u32x4 ragged(const T *p, int have)
{
    constexpr int E = Gran<T>::E;
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = e < have ? Elem<T>::load(p + e) : 0.f;
    return Gran<T>::pack(v);
}

// ---------------------------------------------------------------------------- float32 by bf16 parts

// A float32 is the sum of three bf16: its value rounded, what that leaves rounded, and the rest, which
// fits (G. Henry, P. T. P. Tang, A. Heinecke: Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations, ARITH 2019).  Six of the nine products of two such triples (all but those of 2^-24
// and less) on
// v_mfma_f32_32x32x16_bf16 take three eighths of the float32 instruction's time for the same k-values
// (6 x 32 clocks per 16 of them against 8 x 64).  Their sums are nearer to 64 bits, as the accumulator is
// rounded fewer times: over 32 .. 2048 channels of N(0, 1) values 0.69e-7 .. 7.0e-7 of the result's norm against
// 1.03e-7 .. 8.1e-7.  Three things are looked after:
//   * the bf16 instruction drops what it shifts out, which leaves its sums 1e-8 .. 1e-7 of their norm too
//     low, and that adds up in sums over voxels: half of the results are made with the sign turned (every
//     other voxel; in weight gradients every other split), so that it cancels;
//   * it takes denormal parts and results for zero: both factors are parted 2^24 times as large, at which every bit of a
//     float32, the last of a denormal one too, is a normal bf16, and what falls short as a result is below 2^-173;
//   * infinities, values of 2^104 and products of 2^78 and more leave sums that are not finite: such a tile is made
//     again by the float32 instruction.
// (Instead of the scale, a look at the sums and the largest values for what small values may have lost took 1 to 9 % of
// the kernels, and on volumes with an empty background, where many sums are zero, up to 1.9 times the weight gradients' time:
// 256 x 64 over 80 x 80 x 72 voxels 140 -> 230 us, 128 x 128 43 -> 56; like this 140 and 43.)
static constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;   // (of a factor, of a product)
__device__ inline u32x2 next_part(float (&v)[4])   // four values' next part, which is taken off them
{
    const u32x2 r = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        v[2 * h] -= __uint_as_float(r[h] << 16);
        v[2 * h + 1] -= __uint_as_float(r[h] & 0xffff0000u);
    }
    return r;
}
// A stage of float32 granules in parts: per part, granules of 8 bf16 (two of the float32 ones), four deep;
// the rows turned by four per depth, so that a writer's lanes along the depth do not meet a bank twice.
static const int kPartDepth = 4;
__device__ inline int part_slot(int rows, int part, int d, int r) { return (part * kPartDepth + d) * rows + (r ^ (4 * d)); }
__device__ inline void put_parts(u32x4 *lds, int rows, int q, int r, const float (&g)[4], float scale)
{
    float v[4] = {g[0] * scale, g[1] * scale, g[2] * scale, g[3] * scale};
    u32x2 *half = reinterpret_cast<u32x2 *>(lds);
#pragma unroll
    for (int p = 0; p < 3; ++p) half[2 * part_slot(rows, p, q >> 1, r) + (q & 1)] = next_part(v);
}
// granules of 16 bytes per row of a stage of depth D
template <typename T> constexpr int stage_granules(int depth) { return sizeof(T) == 4 ? 3 * kPartDepth : depth; }
// whether a wavefront's sums are all finite
template <int RT, int CT> __device__ inline bool all_finite(const f32x16 (&acc)[RT][CT])
{
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) t = __builtin_fmaf(acc[i][j][e], 0.f, t);
    return !__any(t != 0.f);
}

// ---------------------------------------------------------------------------- weight gradient

struct WgradParams {
    const void *a, *b;      // (batch, rows, n) and (batch, cols, n)
    float *part;            // split results: (splits, rows * cols + rows), or null with one split
    float *gw, *gb;         // (rows, cols); (rows) or null.  Written here when there is one split
    long long n, chunk;     // voxels per sample; voxels per split, a multiple of a stage's depth
    int rows, cols, tiles_m, tiles_n;
    int per_sample, splits; // splits of a sample; batch * per_sample
};

// Tile of 32 WM RT rows x 32 WN CT columns, WM x WN wavefronts of RT x CT matrix tiles each; a
// stage is D granules deep.  Bound by memory: a 64 x 64 gradient over 2 x 128^3 voxels in bf16 takes
// 0.19 ms (5.6 TB/s on both operands; 0.27 ms as a batch of library GEMMs plus the sum of their
// results), a 64 x 64 one over 183 645 voxels 0.02 ms, a 256 x 64 one 0.04 ms (0.26 ms: the library
// does not split that axis).  What decides is how the loads fall on memory: rows lie megabytes
// apart, so few workgroups with long runs per row (D = 16: 256 bytes) beat many with short ones --
// 512 workgroups, D 16: 192 us; 2048, D 8: 351 us.
// float32: products of bf16 parts (above), parted as they are staged.  256 x 64 over 8 x 16 384 voxels 55 -> 42 us (one
// workgroup's matrix instructions next to the other's parting), 512 x 128 over 8 x 4096 48 -> 37, of which the partial
// results (33 MB written and read) take 14; 32 x 128 over 8 x 65 536, bound by memory, 74 before and after.
template <typename T, int WM, int WN, int RT, int CT, int D>
__global__ void __launch_bounds__(64 * WM * WN, sizeof(T) == 4 ? 2 : 1) wgrad_kernel(WgradParams p)
{
    typedef Gran<T> G;
    constexpr int NT = 64 * WM * WN, BM = 32 * WM * RT, BN = 32 * WN * CT, E = G::E, BK = D * E;
    constexpr int NA = BM * D / NT, NB = BN * D / NT;   // granules a thread stages
    static_assert(NA * NT == BM * D && NB * NT == BN * D, "whole granules per thread");
    constexpr bool F32 = sizeof(T) == 4;
    static_assert(!F32 || D == 2 * kPartDepth, "a stage in parts");
    constexpr int LG = stage_granules<T>(D);
    __shared__ __attribute__((aligned(16))) u32x4 lds[(BM + BN) * LG];
    // an eighth of the launch per XCD (workgroups go round-robin over the eight), the tiles of a split
    // one after the other, so that what they share of the operands comes out of that XCD's L2 (splits
    // dealt to the XCDs whole leave seven of them idle where there is one: 512 x 512 over 64 voxels 8.3
    // us, 5.2 here)
    const int tiles = p.tiles_m * p.tiles_n, total = tiles * p.splits, share = (total + 7) / 8;
    const int index = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
    if (index >= total) return;
    const int tile = index % tiles, split = index / tiles;
    const int m0 = (tile / p.tiles_n) * BM, n0 = (tile % p.tiles_n) * BN;
    const int sample = __builtin_amdgcn_readfirstlane(split / p.per_sample);
    const long long k_lo = (long long)(split % p.per_sample) * p.chunk;
    const long long k_hi = k_lo + p.chunk < p.n ? k_lo + p.chunk : p.n;
    const int tid = threadIdx.x, q = tid % D, r0 = tid / D;
    const T *A = (const T *)p.a + ((long long)sample * p.rows + m0) * p.n;   // (uniform)
    const T *B = (const T *)p.b + ((long long)sample * p.cols + n0) * p.n;
    const bool want_sums = p.gb != nullptr && n0 == 0;
    const float scale = F32 && (split & 1) ? -kScale : kScale;   // (of gz, see above)
    float unscale = split & 1 ? -kUnscale : kUnscale;
    u32x4 ra[NA], rb[NB];
    float sums[NA];

    // Rows past the end repeat the last one: what they contribute is never stored.  Addresses are a
    // uniform pointer plus a 32-bit lane offset (the caller keeps a tile's rows below 4 GiB): as
    // 64-bit lane addresses they took the registers of a third resident wavefront.
    uint32_t off_a[NA], off_b[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i)
        off_a[i] = ((uint32_t)min(r0 + i * (NT / D), p.rows - 1 - m0) * (uint32_t)p.n + q * E) * (uint32_t)sizeof(T);
#pragma unroll
    for (int i = 0; i < NB; ++i)
        off_b[i] = ((uint32_t)min(r0 + i * (NT / D), p.cols - 1 - n0) * (uint32_t)p.n + q * E) * (uint32_t)sizeof(T);
    auto fetch = [&](long long k0) NDC_INLINE {
        const char *a = (const char *)(A + k0), *b = (const char *)(B + k0);
#pragma unroll
        for (int i = 0; i < NA; ++i) ra[i] = *(const u32x4_a2 *)(a + off_a[i]);
#pragma unroll
        for (int i = 0; i < NB; ++i) rb[i] = *(const u32x4_a2 *)(b + off_b[i]);
    };
    auto fetch_ragged = [&](long long k0) NDC_INLINE {
        const char *a = (const char *)(A + k0), *b = (const char *)(B + k0);
        const long long rest = k_hi - k0 - (long long)q * E;
        const int have = rest < 0 ? 0 : rest < E ? (int)rest : E;
#pragma unroll
        for (int i = 0; i < NA; ++i) ra[i] = ragged<T>((const T *)(a + off_a[i]), have);
#pragma unroll
        for (int i = 0; i < NB; ++i) rb[i] = ragged<T>((const T *)(b + off_b[i]), have);
    };
    auto put = [&](auto parts) NDC_INLINE {
        auto store = [&](u32x4 *to, int rows, int r, u32x4 g, float by) NDC_INLINE {
            if constexpr (decltype(parts)::value) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(g[e]);
                put_parts(to, rows, q, r, v, by);
            } else {
                to[slot(rows, q, r)] = g;
            }
        };
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            store(lds, BM, r0 + i * (NT / D), ra[i], scale);
            if (want_sums) sums[i] += G::sum(ra[i]);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) store(lds + BM * LG, BN, r0 + i * (NT / D), rb[i], kScale);
    };

    const int lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN, l32 = lane & 31, kb = lane >> 5;
    f32x16 acc[RT][CT];
    auto multiply = [&](auto parts) NDC_INLINE {
        if constexpr (decltype(parts)::value) {
#pragma unroll
            for (int s = 0; s < kPartDepth / 2; ++s) {
                u32x4 fb[CT][3];
                const int d = 2 * s + kb;
#pragma unroll
                for (int o = 0; o < 3; ++o)
#pragma unroll
                    for (int j = 0; j < CT; ++j) fb[j][o] = lds[BM * LG + part_slot(BN, o, d, 32 * (wn * CT + j) + l32)];
#pragma unroll
                for (int o = 2; o >= 0; --o) {   // the least terms first
                    u32x4 fa[RT];
#pragma unroll
                    for (int i = 0; i < RT; ++i) fa[i] = lds[part_slot(BM, o, d, 32 * (wm * RT + i) + l32)];
#pragma unroll
                    for (int b = 2 - o; b >= 0; --b)
#pragma unroll
                        for (int i = 0; i < RT; ++i)
#pragma unroll
                            for (int j = 0; j < CT; ++j) acc[i][j] = Gran<bf16_t>::mma(fa[i], fb[j][b], acc[i][j]);
                }
            }
        } else {
#pragma unroll
            for (int s = 0; s < D / 2; ++s) {
                u32x4 fa[RT], fb[CT];
                const int d = 2 * s + kb;
#pragma unroll
                for (int i = 0; i < RT; ++i) fa[i] = lds[slot(BM, d, 32 * (wm * RT + i) + l32)];
#pragma unroll
                for (int j = 0; j < CT; ++j) fb[j] = lds[BM * LG + slot(BN, d, 32 * (wn * CT + j) + l32)];
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < CT; ++j) acc[i][j] = G::mma(fa[i], fb[j], acc[i][j]);
            }
        }
    };
    // Whole stages in a loop without conditions: the next stage's loads are in flight while this
    // one multiplies.  (A branch between the two forms of fetch inside the loop made every stage
    // wait for its loads before it multiplied.)
    auto clear = [&]() NDC_INLINE {
#pragma unroll
        for (int i = 0; i < NA; ++i) sums[i] = 0.f;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = f32x16{};
    };
    auto last = [&](long long k0, auto parts) NDC_INLINE {
        fetch_ragged(k0);
        put(parts);
        __syncthreads();
        multiply(parts);
    };
    clear();
    const std::bool_constant<F32> parts;
    const int stages = (int)((k_hi - k_lo) / BK);
    if (stages > 0) fetch(k_lo);
    for (int s = 0; s < stages; ++s) {
        put(parts);
        __syncthreads();
        fetch(k_lo + (long long)(s + 1 < stages ? s + 1 : s) * BK);
        multiply(parts);
        __syncthreads();
    }
    if (k_lo + (long long)stages * BK < k_hi) last(k_lo + (long long)stages * BK, parts);
    if constexpr (F32) {
        __shared__ int finite[WM * WN];
        if (const bool f = all_finite(acc); lane == 0) finite[wave] = f;
        __syncthreads();
        bool again = false;
#pragma unroll
        for (int w = 0; w < WM * WN; ++w) again = again || !finite[w];
        if (__builtin_expect(again, 0)) {
            clear();
            unscale = 1.f;
            for (long long k0 = k_lo; k0 < k_hi; k0 += BK) {
                last(k0, std::false_type());
                __syncthreads();
            }
        }
    }
    const long long out_size = (long long)p.rows * p.cols;
    float *gw = p.part ? p.part + split * (out_size + p.rows) : p.gw;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const int col = n0 + 32 * (wn * CT + j) + l32;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + 32 * (wm * RT + i) + 8 * (e / 4) + 4 * kb + e % 4;
                if (row < p.rows && col < p.cols)
                    gw[(long long)row * p.cols + col] = F32 ? acc[i][j][e] * unscale : acc[i][j][e];
            }
        }
    if (want_sums) {
        float *gb = p.part ? p.part + split * (out_size + p.rows) + out_size : p.gb;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            float s = sums[i];
#pragma unroll
            for (int o = 1; o < D; o *= 2) s += __shfl_xor(s, o);
            const int row = m0 + r0 + i * (NT / D);
            if (q == 0 && row < p.rows) gb[row] = s;
        }
    }
}

// The same over few voxels: one workgroup has a TL x TL tile of the result and all voxels, its sixteen
// wavefronts take turns of 64 / TL granules and their results are added through LDS.  No splits, hence no
// partial results and no second launch to add them: what these sizes cost is launches and the latency of
// one, and between two launches of a recorded step lie 1-2 us besides.  Tiles of 16 as long as that
// gives each CU one: it multiplies 1024 voxels of a 32 x 32 tile in float32 in 3.4 us.
// MANY: the turns of all samples are one count, of which each wavefront has four in flight; one sample after the
// other, 64 samples of 16 voxels waited 64 times (32 x 32 in bf16, with the projection itself, 94 us; 21 like this).
// For few samples the plain loops are the shorter code: 32 x 32 over 2 x 250 in float32 7.0 us against 7.8.
static const int kWholeWaves = 16;
template <typename T, int TL, bool MANY> __global__ void __launch_bounds__(64 * kWholeWaves) wgrad_whole_kernel(WgradParams p)
{
    typedef Gran<T> G;
    typedef std::conditional_t<TL == 32, f32x16, f32x4> Acc;
    constexpr int E = G::E, NW = kWholeWaves, Q = 64 / TL, NE = TL * TL / 64;
    __shared__ float acc_lds[NW][TL * TL];
    __shared__ float sum_lds[NW][64];
    const int m0 = (int)(blockIdx.x / p.tiles_n) * TL, n0 = (int)(blockIdx.x % p.tiles_n) * TL;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane % TL, kb = lane / TL;
    const bool want_sums = p.gb != nullptr && n0 == 0;
    // (rows past the end repeat the last one: what they contribute is never stored)
    const T *a = (const T *)p.a + (long long)min(m0 + l, p.rows - 1) * p.n + kb * E;
    const T *b = (const T *)p.b + (long long)min(n0 + l, p.cols - 1) * p.n + kb * E;
    const int full = (int)(p.n / (Q * E));
    Acc acc = Acc{};
    float sum = 0.f;
    auto add = [&](u32x4 fa, u32x4 fb) {
        if (want_sums) sum += G::sum(fa);
        acc = G::mma(fa, fb, acc);
    };
    if constexpr (MANY) {
        const int turns = (int)((p.n + Q * E - 1) / (Q * E)), total = p.splits * turns;
        for (int k = wave; k < total; k += 4 * NW) {
            u32x4 fa[4], fb[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int at = k + u * NW, s = at / turns, i = at - s * turns;
                fa[u] = fb[u] = u32x4{};
                if (at >= total) continue;
                const T *as = a + (long long)s * p.rows * p.n + i * Q * E, *bs = b + (long long)s * p.cols * p.n + i * Q * E;
                if (i < full) {
                    fa[u] = *(const u32x4_a2 *)as;
                    fb[u] = *(const u32x4_a2 *)bs;
                } else {   // voxels past the whole turns
                    const int rest = (int)p.n - (i * Q + kb) * E, have = rest < 0 ? 0 : rest < E ? rest : E;
                    fa[u] = ragged<T>(as, have);
                    fb[u] = ragged<T>(bs, have);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k + u * NW < total) add(fa[u], fb[u]);
        }
    } else {
        for (int s = 0; s < p.splits; ++s) {   // samples
            const T *as = a + (long long)s * p.rows * p.n, *bs = b + (long long)s * p.cols * p.n;
            int i = wave;
            for (; i + 3 * NW < full; i += 4 * NW) {
                u32x4 fa[4], fb[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    fa[u] = *(const u32x4_a2 *)(as + (i + u * NW) * Q * E);
                    fb[u] = *(const u32x4_a2 *)(bs + (i + u * NW) * Q * E);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) add(fa[u], fb[u]);
            }
            for (; i < full; i += NW) add(*(const u32x4_a2 *)(as + i * Q * E), *(const u32x4_a2 *)(bs + i * Q * E));
            if (i == full && p.n % (Q * E)) {   // voxels past the whole turns
                const int rest = (int)p.n - (i * Q + kb) * E, have = rest < 0 ? 0 : rest < E ? rest : E;
                add(ragged<T>(as + i * Q * E, have), ragged<T>(bs + i * Q * E, have));
            }
        }
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) acc_lds[wave][e * 64 + lane] = acc[e];
    if (want_sums) sum_lds[wave][lane] = sum;
    __syncthreads();
    const int e = threadIdx.x >> 6;
    if (e < NE) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += acc_lds[w][threadIdx.x];
        const int row = m0 + (TL == 32 ? 8 * (e / 4) + 4 * kb + e % 4 : 4 * kb + e), col = n0 + l;
        if (row < p.rows && col < p.cols) p.gw[(long long)row * p.cols + col] = v;
    }
    if (want_sums && threadIdx.x < TL && m0 + (int)threadIdx.x < p.rows) {
        float t = 0.f;
        for (int w = 0; w < NW; ++w)
#pragma unroll
            for (int q = 0; q < Q; ++q) t += sum_lds[w][threadIdx.x + q * TL];
        p.gb[m0 + threadIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------- y = epilogue(W x)

struct TileParams {
    const void *x;           // (batch, cin, n)
    const float *w;          // W (cout, cin), or (cin, cout) storage of it
    const float *bias;       // cout values or null
    const void *res;         // (batch, cout, n) or null: added to y; with a gradient mode the
                             // pre-activation whose derivative (at res + bias) multiplies the product
    const void *mask;        // (batch, cout, n) or null: y is zero where mask <= 0
    void *y, *zkeep;         // (batch, cout, n); zkeep or null: the product before bias and activation
    float *gpart;            // kGeluGrad: (voxel tiles, cout) sums of y over a tile's voxels, or null
    long long n;
    int cin, cout, tiles_m, tiles_n, batch;
};

// modes: epilogue::kNone / kRelu / kGelu, and the product times the GELU's derivative
enum { kGeluGrad = 4 };

template <typename T> struct Quad;   // 4 voxels of one row
template <> struct Quad<float> {
    f32x4 v;
    __device__ float get(int i) const { return v[i]; }
    __device__ void load(const float *p) { v = __builtin_bit_cast(f32x4, *(const u32x4_a2 *)p); }
    __device__ void store(float *p) const { *(u32x4_a2 *)p = __builtin_bit_cast(u32x4, v); }
    __device__ void set(const float (&f)[4]) { v = f32x4{f[0], f[1], f[2], f[3]}; }
};
template <> struct Quad<bf16_t> {
    u32x2 v;
    __device__ float get(int i) const
    {
        const uint32_t w = v[i >> 1];
        return __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
    }
    __device__ void load(const bf16_t *p) { v = *(const u32x2_a2 *)p; }
    __device__ void store(bf16_t *p) const { *(u32x2_a2 *)p = v; }
    __device__ void set(const float (&f)[4]) { v = u32x2{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])}; }
};

template <typename T> __device__ inline Quad<T> load_quad(const T *p, int have)
{
    Quad<T> r;
    if (have >= 4) {
        r.load(p);
    } else {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = i < have ? Elem<T>::load(p + i) : 0.f;
        r.set(v);
    }
    return r;
}
template <typename T> __device__ inline void store_quad(T *p, const float (&f)[4], int have)
{
    if (have >= 4) {
        Quad<T> r;
        r.set(f);
        r.store(p);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < have) Elem<T>::store(p + i, f[i]);
    }
}

// (8 rows of k) x (4 voxels) -> four granules
__device__ inline void transpose(const Quad<bf16_t> (&in)[8], u32x4 (&out)[4])
{
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) {
            out[2 * h][pr] = __builtin_amdgcn_perm(in[2 * pr + 1].v[h], in[2 * pr].v[h], 0x05040100u);
            out[2 * h + 1][pr] = __builtin_amdgcn_perm(in[2 * pr + 1].v[h], in[2 * pr].v[h], 0x07060302u);
        }
}

// The epilogue of NR consecutive rows of four voxels: z the products, `have` of the four voxels
// exist (`whole`: all of them, in every lane).  What it reads is requested ahead of its stores.
// sums (kGeluGrad): each row's sum over the voxels that exist, of the float32 values before they
// are stored -- the bias gradient is these, and must not carry the rounding of what is stored.
template <typename T, int MODE, int NR>
__device__ inline void finish(const TileParams &p, const float (&z)[NR][4], int row0, long long base, int have, bool whole,
                              float (&sums)[NR])
{
#pragma unroll
    for (int e = 0; e < NR; ++e) sums[e] = 0.f;
    auto run = [&](auto tag) {
        constexpr bool WHOLE = decltype(tag)::value;
        Quad<T> rq[NR], mq[NR];
        float bias[NR];
#pragma unroll
        for (int e = 0; e < NR; ++e) {
            const int row = min(row0 + e, p.cout - 1);
            const long long at = base + (long long)row * p.n;
            bias[e] = p.bias ? p.bias[row] : 0.f;
            if (p.res) rq[e] = load_quad<T>((const T *)p.res + at, WHOLE ? 4 : have);
            if (p.mask) mq[e] = load_quad<T>((const T *)p.mask + at, WHOLE ? 4 : have);
        }
#pragma unroll
        for (int e = 0; e < NR; ++e) {
            if (row0 + e >= p.cout) continue;
            const long long at = base + (long long)(row0 + e) * p.n;
            float y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (MODE == kGeluGrad) {
                    y[j] = z[e][j] * epilogue::act_grad<epilogue::kGelu>(rq[e].get(j) + bias[e]);
                    sums[e] += WHOLE || j < have ? y[j] : 0.f;
                } else {
                    y[j] = epilogue::act_fwd<MODE>(z[e][j] + bias[e]);
                    if (p.res) y[j] += rq[e].get(j);
                    if (p.mask) y[j] = mq[e].get(j) > 0.f ? y[j] : 0.f;
                }
            }
            if constexpr (MODE == epilogue::kRelu || MODE == epilogue::kGelu)
                if (p.zkeep) store_quad<T>((T *)p.zkeep + at, z[e], WHOLE ? 4 : have);
            store_quad<T>((T *)p.y + at, y, WHOLE ? 4 : have);
        }
    };
    if (whole) run(std::true_type{});
    else run(std::false_type{});
}

// bf16: a workgroup of WAVES wavefronts makes a tile of 32 WAVES output rows x 128 voxels.  Voxel
// v of the tile is column v / 4 of matrix tile v % 4, so that a lane ends up with four
// consecutive voxels of a row: stores (and the loads of residual, mask and kept product) are 8
// or 16 bytes per lane, 32 lanes contiguous.
template <bool WT, int WAVES, int MODE>
__global__ void __launch_bounds__(64 * WAVES) tile_kernel(TileParams p)
{
    typedef bf16_t T;
    typedef Gran<T> G;
    constexpr int NT = 64 * WAVES, BM = 32 * WAVES, BN = 128, E = G::E, BK = kDepth * E;
    constexpr int NA = BM * kDepth / NT;             // weight granules a thread stages
    constexpr int NB = 32 * kDepth / NT;             // voxel quads a thread stages
    static_assert(NA * NT == BM * kDepth && NB * NT == 32 * kDepth, "whole granules per thread");
    __shared__ __attribute__((aligned(16))) u32x4 lds[(BM + BN) * kDepth];
    const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3;
    const int tile_m = pos % p.tiles_m, vt = (pos / p.tiles_m) * 8 + xcd;   // a voxel tile stays on one XCD
    if (vt >= p.tiles_n * p.batch) return;
    const int sample = vt / p.tiles_n, m0 = tile_m * BM;
    const long long v0 = (long long)(vt % p.tiles_n) * BN;
    const int tid = threadIdx.x;
    const T *X = (const T *)p.x + (long long)sample * p.cin * p.n + v0;
    const float *W = p.w;
    const int left = (int)(p.n - v0 < BN ? p.n - v0 : BN);   // voxels of this tile

    float rw[NA][E];
    Quad<T> rx[NB][E];
    auto weight_at = [&](int i, int &r, int &q) {   // granule i of this thread
        const int g = tid + i * NT;
        if (WT) r = g % BM, q = g / BM;             // lanes along the rows of W, contiguous in W^T
        else r = g >> 3, q = g & 7;
    };
    // Whole granules and quads (all but the narrow first layers and the last voxel tile of an odd
    // count): loads without conditions, and nothing done to their values before `put`, so that a
    // stage's loads stay in flight while the stage before it multiplies.  Rows and quads past the
    // end repeat the last one -- their results are never stored --, depths past the end are zeroed.
    const bool whole = p.cin % E == 0 && left % 4 == 0;
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            int r, q;
            weight_at(i, r, q);
            const int m = min(m0 + r, p.cout - 1), k = min(k0 + q * E, p.cin - E);
            if constexpr (WT) {
#pragma unroll
                for (int e = 0; e < E; ++e) rw[i][e] = W[(long long)(k + e) * p.cout + m];
            } else {
#pragma unroll
                for (int h = 0; h < E / 4; ++h) {
                    Quad<float> t;
                    t.load(W + (long long)m * p.cin + k + 4 * h);
#pragma unroll
                    for (int e = 0; e < 4; ++e) rw[i][4 * h + e] = t.get(e);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int u = tid + i * NT, c = min(u & 31, left / 4 - 1), k = min(k0 + (u >> 5) * E, p.cin - E);
            const T *src = X + (long long)k * p.n + 4 * c;
#pragma unroll
            for (int e = 0; e < E; ++e) rx[i][e].load(src + (long long)e * p.n);
        }
    };
    auto fetch_ragged = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            int r, q;
            weight_at(i, r, q);
            const int m = m0 + r, k = k0 + q * E, have = m < p.cout ? p.cin - k : 0;
#pragma unroll
            for (int e = 0; e < E; ++e)
                rw[i][e] = e < have ? W[WT ? (long long)(k + e) * p.cout + m : (long long)m * p.cin + k + e] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int u = tid + i * NT, c = u & 31, k = k0 + (u >> 5) * E;
            const T *src = X + (long long)k * p.n + 4 * c;
#pragma unroll
            for (int e = 0; e < E; ++e)
                rx[i][e] = load_quad<T>(src + (long long)e * p.n, k + e < p.cin ? left - 4 * c : 0);
        }
    };
    auto put = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            int r, q;
            weight_at(i, r, q);
            const uint32_t keep = k0 + q * E < p.cin ? ~0u : 0u;
            u32x4 g = G::pack(rw[i]);
#pragma unroll
            for (int e = 0; e < 4; ++e) g[e] &= keep;
            lds[slot(BM, q, r)] = g;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int u = tid + i * NT, c = u & 31, q = u >> 5;
            const uint32_t keep = k0 + q * E < p.cin ? ~0u : 0u;
            u32x4 g[4];
            transpose(rx[i], g);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e) g[j][e] &= keep;
                lds[BM * kDepth + slot(BN, q, 32 * j + c)] = g[j];
            }
        }
    };

    const int lane = tid & 63, wave = tid >> 6, l32 = lane & 31, kb = lane >> 5;
    f32x16 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x16{};
    auto multiply = [&](int k0) {
        const int steps = p.cin - k0 >= BK ? kDepth / 2 : (p.cin - k0 + 2 * E - 1) / (2 * E);
        for (int s = 0; s < steps; ++s) {
            const int d = 2 * s + kb;
            const u32x4 fa = lds[slot(BM, d, 32 * wave + l32)];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = G::mma(fa, lds[BM * kDepth + slot(BN, d, 32 * j + l32)], acc[j]);
        }
    };
    if (whole) {
        fetch(0);
        for (int k0 = 0; k0 < p.cin; k0 += BK) {
            put(k0);
            __syncthreads();
            if (k0 + BK < p.cin) fetch(k0 + BK);
            multiply(k0);
            __syncthreads();
        }
    } else {
        for (int k0 = 0; k0 < p.cin; k0 += BK) {
            fetch_ragged(k0);
            put(k0);
            __syncthreads();
            multiply(k0);
            __syncthreads();
        }
    }
    const int have = left - 4 * l32;
    const bool summed = MODE == kGeluGrad && p.gpart != nullptr;   // (then every lane takes part below)
    if (have <= 0 && !summed) return;
    const long long base = (long long)sample * p.cout * p.n + v0 + 4 * l32;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        float z[4][4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < 4; ++j) z[e][j] = acc[j][4 * h + e];
        const int row0 = m0 + 32 * wave + 8 * h + 4 * kb;
        float sums[4] = {0.f, 0.f, 0.f, 0.f};
        if (have > 0) finish<T, MODE, 4>(p, z, row0, base, have, whole, sums);
        if (summed) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float s = epilogue::half_sum(sums[e]);   // the 32 lanes of a row
                if (l32 == 31 && row0 + e < p.cout) p.gpart[(long long)vt * p.cout + row0 + e] = s;
            }
        }
    }
}

// float32: a workgroup of four wavefronts makes 32 RT output rows x 128 voxels, each wavefront all of the rows of
// 32 voxels.  The products are those of bf16 parts (above).  A wavefront's voxels are its own, so x goes from
// memory to its registers and is parted there, a word per lane and channel; only W, which the wavefronts share,
// is parted into LDS, in two buffers, one barrier per 32 channels.  (With x through LDS as well, parting and
// staging took as long as the matrix instructions: 128 -> 512 channels over 8 x 4096 voxels 41 us.)
// CHAINS: the sums of 32 channels are made apart and then added, which keeps the error of any number of channels
// below that of the sliced form (2048 channels 1.7e-7 of the result's norm instead of 7.0e-7; slices 2.9e-7).  It
// takes a wavefront per SIMD: without it 32 -> 128 over 8 x 65 536 takes 77 us instead of 85, 64 -> 256 over
// 8 x 16 384 43 instead of 49, with 0.69e-7 and 1.1e-7 (the float32 instruction: 1.03e-7, 1.45e-7).
// Bound by memory to 64 channels (64 -> 256 over 8 x 16 384: 4.0 TB/s), beyond by the matrix instructions,
// which run at 45 clocks each at the clock that their power leaves, and the vector instructions that part x and W
// between them: 512 -> 128 over 8 x 4096 78 us by the float32 instruction, 34 like this; 256 -> 1024 over 8 x 1024
// 45 and 35; 256 -> 64 over 8 x 16 384 50 and 36; 96 -> 64 over 33 333 23 and 11.
template <bool WT, int RT, bool CHAINS, int MODE>
__global__ void __launch_bounds__(256, (RT == 2 ? 4 : 5) - CHAINS) parts_kernel(TileParams p)
{
    constexpr int BM = 32 * RT, BN = 128, BK = 32;
    __shared__ __attribute__((aligned(16))) u32x4 lds[2][BM * 3 * kPartDepth];
    __shared__ __attribute__((aligned(16))) float bias[BM];
    __shared__ float red[4][BM];
    const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3;
    const int tile_m = pos % p.tiles_m, vt = (pos / p.tiles_m) * 8 + xcd;   // a voxel tile stays on one XCD
    if (vt >= p.tiles_n * p.batch) return;
    const int sample = vt / p.tiles_n, m0 = tile_m * BM;
    const long long v0 = (long long)(vt % p.tiles_n) * BN;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, kb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int left = (int)(p.n - v0 < BN ? p.n - v0 : BN), mine = 32 * wave + l32;
    const float *X = (const float *)p.x + (long long)sample * p.cin * p.n + v0;
    // lanes past the end of a row repeat its last voxel, rows past the end the last row: never stored
    const uint32_t xoff = ((uint32_t)(8 * kb) * (uint32_t)p.n + (uint32_t)min(mine, left - 1)) * 4u;
    const float scale = l32 & 1 ? -kScale : kScale;
    float xr[2][8], rw[RT][4];
    auto weight_at = [&](int i, int &r, int &q) NDC_INLINE {   // granule i of this thread
        const int g = tid + i * 256;
        if (WT) r = g % BM, q = g / BM;   // lanes along the rows of W, contiguous in W^T
        else r = g >> 3, q = g & 7;
    };
    auto fetch = [&](int k0) NDC_INLINE {   // (whole stages)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 8; ++e) xr[t][e] = *(const float *)((const char *)(X + (long long)(k0 + 16 * t + e) * p.n) + xoff);
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            int r, q;
            weight_at(i, r, q);
            const int m = min(m0 + r, p.cout - 1), k = k0 + 4 * q;
            if constexpr (WT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) rw[i][e] = p.w[(long long)(k + e) * p.cout + m];
            } else {
                Quad<float> t;
                t.load(p.w + (long long)m * p.cin + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) rw[i][e] = t.get(e);
            }
        }
    };
    auto fetch_ragged = [&](int k0) NDC_INLINE {   // (depths past the end are zero)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = k0 + 16 * t + 8 * kb + e;
                xr[t][e] = k < p.cin ? X[(long long)k * p.n + min(mine, left - 1)] : 0.f;
            }
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            int r, q;
            weight_at(i, r, q);
            const int m = min(m0 + r, p.cout - 1), k = k0 + 4 * q;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                rw[i][e] = k + e < p.cin ? p.w[WT ? (long long)(k + e) * p.cout + m : (long long)m * p.cin + k + e] : 0.f;
        }
    };
    f32x16 acc[RT][1];
    u32x4 xp[2][1][3];
    // halves: 2, or 1 in a last stage of 16 channels and fewer (us, 16 -> 64 over 98 x 1000 voxels 13.8 with both, 12.5 with one;
    // with 32 rows the choice costs registers that are not there, 22 -> 29 for 32 channels)
    auto put = [&](u32x4 *to, int halves) NDC_INLINE {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            int r, q;
            weight_at(i, r, q);
            put_parts(to, BM, q, r, rw[i], kScale);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (t >= halves) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = xr[t][4 * h + e] * scale;
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    const u32x2 w = next_part(v);
                    xp[t][0][o][2 * h] = w[0], xp[t][0][o][2 * h + 1] = w[1];
                }
            }
        }
    };
    auto multiply = [&](const u32x4 *from, int halves) NDC_INLINE {
        f32x16 sum[RT];
        if constexpr (!CHAINS) {
#pragma unroll
            for (int i = 0; i < RT; ++i) sum[i] = acc[i][0];
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (t >= halves) continue;
#pragma unroll
            for (int o = 2; o >= 0; --o) {   // the least terms first
                u32x4 fa[RT];
#pragma unroll
                for (int i = 0; i < RT; ++i) fa[i] = from[part_slot(BM, o, 2 * t + kb, 32 * i + l32)];
#pragma unroll
                for (int b = 2 - o; b >= 0; --b)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        sum[i] = Gran<bf16_t>::mma(fa[i], xp[t][0][b], CHAINS && t == 0 && o == 2 ? f32x16{} : sum[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i][0] = CHAINS ? acc[i][0] + sum[i] : sum[i];
    };
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i][0] = f32x16{};
    for (int r = tid; r < BM; r += 256) bias[r] = p.bias && m0 + r < p.cout ? p.bias[m0 + r] : 0.f;
    const int stages = p.cin / BK;
    if (stages > 0) fetch(0);
    for (int s = 0; s < stages; ++s) {
        put(lds[s & 1], 2);
        __syncthreads();
        if (s + 1 < stages) fetch((s + 1) * BK);
        multiply(lds[s & 1], 2);
    }
    if (stages * BK < p.cin) {
        fetch_ragged(stages * BK);
        const int halves = RT == 2 && p.cin - stages * BK <= 16 ? 1 : 2;
        put(lds[stages & 1], halves);
        __syncthreads();
        multiply(lds[stages & 1], halves);
    }
    float unscale = l32 & 1 ? -kUnscale : kUnscale;
    if (__builtin_expect(!all_finite(acc), 0)) {
        unscale = 1.f;
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i][0] = f32x16{};
        for (int k0 = 0; k0 < p.cin; k0 += 2) {
            const int k = k0 + kb;
            const bool in = k < p.cin;
            const float b = in ? X[(long long)k * p.n + min(mine, left - 1)] : 0.f;
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int m = min(m0 + 32 * i + l32, p.cout - 1);
                const float a = in ? p.w[WT ? (long long)k * p.cout + m : (long long)m * p.cin + k] : 0.f;
                acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i][0], 0, 0, 0);
            }
        }
    }
    const bool summed = MODE == kGeluGrad && p.gpart != nullptr, exists = mine < left;
    const long long base = ((long long)sample * p.cout + m0) * p.n + v0;   // (uniform)
    const uint32_t yoff = ((uint32_t)(4 * kb) * (uint32_t)p.n + (uint32_t)min(mine, left - 1)) * 4u;
    auto run = [&](auto tag) NDC_INLINE {
        constexpr bool WHOLE = decltype(tag)::value;   // all rows and voxels of the tile exist
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {   // what eight rows read is requested ahead of their stores
                float rv[8], mv[8], bv[8];
                auto row_of = [&](int e) NDC_INLINE { return 32 * i + 16 * h + 8 * (e / 4) + e % 4; };   // (+ 4 kb)
                auto in = [&](int e) NDC_INLINE { return WHOLE || (exists && m0 + row_of(e) + 4 * kb < p.cout); };
                auto at = [&](const void *t, int e) NDC_INLINE {
                    return (float *)((char *)((float *)t + base + (long long)row_of(e) * p.n) + yoff);
                };
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    bv[e] = bias[row_of(e) + 4 * kb];
                    if (p.res) rv[e] = in(e) ? *at(p.res, e) : 0.f;
                    if (p.mask) mv[e] = in(e) ? *at(p.mask, e) : 0.f;
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float z = acc[i][0][8 * h + e] * unscale;
                    float y;
                    if constexpr (MODE == kGeluGrad) {
                        y = z * epilogue::act_grad<epilogue::kGelu>(rv[e] + bv[e]);
                    } else {
                        y = epilogue::act_fwd<MODE>(z + bv[e]);
                        if (p.res) y += rv[e];
                        if (p.mask) y = mv[e] > 0.f ? y : 0.f;
                    }
                    if (in(e)) {
                        if constexpr (MODE == epilogue::kRelu || MODE == epilogue::kGelu)
                            if (p.zkeep) *at(p.zkeep, e) = z;
                        *at(p.y, e) = y;
                    }
                    if (summed) {
                        const float sum = epilogue::half_sum(in(e) ? y : 0.f);   // the 32 lanes of a row
                        if (l32 == 31) red[wave][row_of(e) + 4 * kb] = sum;
                    }
                }
            }
    };
    if (left == BN && m0 + BM <= p.cout) run(std::true_type{});
    else run(std::false_type{});
    if (summed) {
        __syncthreads();
        if (tid < BM && m0 + tid < p.cout)
            p.gpart[(long long)vt * p.cout + m0 + tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
    }
}

// ---------------------------------------------------------------------------- small grids

// A grid of a few thousand voxels leaves the tiled kernel a handful of workgroups that walk the
// channels one stage after the other, each stage waiting for memory (2048 -> 512 channels over
// 64 voxels: 32 stages, 195 us).  Here the channels are split over the wavefronts of a workgroup
// instead: a tile is R output rows x 2 R voxels, wavefront w takes its share of the channels
// straight from memory into the operand registers (AHEAD steps requested together, no staging,
// no barrier), and the wavefronts' partial tiles are added through LDS, in order.  Lanes hold
// voxel pairs: pair c is column c of an even-voxel and an odd-voxel matrix tile.
// R = 16 where 32 x 64 tiles would leave CUs without one: what bounds such a launch is the matrix
// work and the round trips to memory of the few workgroups there are (2048 -> 512 channels over 143
// voxels in float32: 48 tiles of 14 us of matrix instructions each), so four times the tiles, each
// with a quarter of the products and half as many round trips.  (The 2-D network's projections over
// 143 and 572 voxels: 13-23 -> 9-13 us.)
static const int kMaxSlices = 8;

template <typename T, bool WT, int MODE, int R>
__global__ void __launch_bounds__(64 * kMaxSlices) sliced_kernel(TileParams p)
{
    typedef Gran<T> G;
    typedef typename std::conditional<R == 16, f32x4, f32x16>::type Acc;
    constexpr int E = G::E, KB = 64 / R;             // granules of a step
    constexpr int kAhead = R == 16 && E == 4 ? 8 : 4;   // steps whose operands are in flight
    __shared__ __attribute__((aligned(16))) float part[kMaxSlices][R][2 * R];
    // an eighth of the tiles per XCD, consecutive ones, so that the voxel tiles of a row tile, which
    // read the same rows of W, share an L2 (whole row tiles dealt to the XCDs leave all but a few of
    // them idle where there are fewer than eight: 128 -> 32 channels over 36 608 voxels 45 us, 10 here)
    const int vts = p.tiles_n * p.batch, tiles = p.tiles_m * vts, share = (tiles + 7) / 8;
    const int index = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
    if (index >= tiles) return;
    const int tile_m = index / vts, vt = index % vts;
    const int sample = vt / p.tiles_n, m0 = tile_m * R;
    const int v0 = (vt % p.tiles_n) * 2 * R, left = min((int)p.n - v0, 2 * R);
    const int tid = threadIdx.x, lane = tid & 63, col = lane % R, kb = lane / R, slices = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T *X = (const T *)p.x + (long long)sample * p.cin * p.n + v0;
    const int m = min(m0 + col, p.cout - 1);
    // pairs past the end repeat the last one; the half pair at the end of an odd count is the
    // second element of the pair before it
    const bool half = 2 * col + 1 == left;
    const int c = min(2 * col, left - 2);   // (-1 in a tile of one voxel: n >= 2)
    const int steps = (p.cin + KB * E - 1) / (KB * E), per = (steps + slices - 1) / slices;
    const int s_lo = wave * per, s_hi = min(s_lo + per, steps);
    typedef typename std::conditional<sizeof(T) == 2, uint32_t, u32x2>::type Pair;   // two voxels
    typedef Pair Pair_a2 __attribute__((aligned(2), may_alias));
    float w[kAhead][E];
    Pair xv[kAhead][E];
    auto request = [&](int a, int s) {
        const int k = min((KB * s + kb) * E, p.cin - E);   // (the caller has checked cin % E == 0, n >= 2)
        if constexpr (WT) {
#pragma unroll
            for (int e = 0; e < E; ++e) w[a][e] = p.w[(long long)(k + e) * p.cout + m];
        } else {
#pragma unroll
            for (int h = 0; h < E / 4; ++h) {
                Quad<float> t;
                t.load(p.w + (long long)m * p.cin + k + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e) w[a][4 * h + e] = t.get(e);
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) xv[a][e] = *(const Pair_a2 *)(X + (long long)(k + e) * p.n + c);
    };
    Acc acc0 = {}, acc1 = {};
    const uint32_t second = half ? ~0u : 0u;
    auto multiply = [&](int a, int s) {
        // (masks instead of selects: a condition here becomes a branch around the loads' first use)
        const uint32_t keep = (KB * s + kb) * E < p.cin ? ~0u : 0u;
        u32x4 gw = G::pack(w[a]), g0, g1;
        if constexpr (sizeof(T) == 2) {
#pragma unroll
            for (int pr = 0; pr < 4; ++pr) {
                const uint32_t e0 = xv[a][2 * pr] >> (second & 16u), e1 = xv[a][2 * pr + 1] >> (second & 16u);
                g0[pr] = __builtin_amdgcn_perm(e1, e0, 0x05040100u) & keep;
                g1[pr] = __builtin_amdgcn_perm(xv[a][2 * pr + 1], xv[a][2 * pr], 0x07060302u) & keep;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g0[e] = ((xv[a][e][0] & ~second) | (xv[a][e][1] & second)) & keep;
                g1[e] = xv[a][e][1] & keep;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) gw[e] &= keep;
        acc0 = G::mma(gw, g0, acc0);
        acc1 = G::mma(gw, g1, acc1);
    };
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
        if (s_lo + a < s_hi) request(a, s_lo + a);
    for (int s0 = s_lo; s0 < s_hi; s0 += kAhead) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            if (s0 + a < s_hi) multiply(a, s0 + a);
            if (s0 + a + kAhead < s_hi) request(a, s0 + a + kAhead);
        }
    }
#pragma unroll
    for (int j = 0; j < R * R / 64; ++j)   // (a lane has runs of four rows, 4 KB rows apart)
        *reinterpret_cast<float2 *>(&part[wave][4 * KB * (j / 4) + 4 * kb + j % 4][2 * col]) = make_float2(acc0[j], acc1[j]);
    __syncthreads();
    const bool summed = MODE == kGeluGrad && p.gpart != nullptr;
    for (int t = tid; t < R * R / 2; t += blockDim.x) {   // (whole wavefronts: both counts are multiples of 64)
        const int row = t / (R / 2), q = t % (R / 2), have = left - 4 * q;
        const bool mine = m0 + row < p.cout && have > 0;
        if (!mine && !summed) continue;
        float sums[1] = {0.f};
        if (mine) {
            float z[1][4] = {{0.f, 0.f, 0.f, 0.f}};
            for (int w = 0; w < slices; ++w) {
                const float4 v = *reinterpret_cast<const float4 *>(&part[w][row][4 * q]);
                z[0][0] += v.x, z[0][1] += v.y, z[0][2] += v.z, z[0][3] += v.w;
            }
            finish<T, MODE, 1>(p, z, m0 + row, (long long)sample * p.cout * p.n + v0 + 4 * q, have, false, sums);
        }
        if (summed) {
            float s = sums[0];
#pragma unroll
            for (int o = 1; o < R / 2; o *= 2) s += __shfl_xor(s, o);   // the lanes of a row
            if (q == 0 && m0 + row < p.cout) p.gpart[(long long)vt * p.cout + m0 + row] = s;
        }
    }
}

}  // namespace gemm
}  // namespace ndc
