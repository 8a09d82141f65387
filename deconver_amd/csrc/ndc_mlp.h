// The MLP of a Deconver block on channel-first bf16 tensors with its hidden tensor on chip,
//
//   y = W2 gelu(W1 x + b1) + b2 + residual            W1: 4C x C, W2: C x 4C, C = 32 or 64
//
// (layers/mlp.py:40-63 of the reference with the block's sum, deconver.py:60-64), and its backward,
// which forms the hidden tensor again from x:
//
//   u = W1 x + b1,  h = gelu(u),  gu = (W2^T gy) * gelu'(u),  gx = W1^T gu,
//   gW1 = gu x^T,  gW2 = gy h^T,  gb1 = sum gu (before its rounding),  gb2 = sum gy.
//
// Why: as two projections the 4C-channel hidden tensor is written twice (product and GELU) and read
// once in the forward and written once and read four times in the backward, 39 passes over a C-channel
// tensor; here the forward moves 3 and the backward 3, and its up to 256 workgroups' partial weight
// gradients, which a second launch adds: 34 MB written and read at C = 64 (a pass over 266 000 voxels), 8.6 at 32.
// What bounds both is then the GELU on the vector unit (two transcendental and a dozen other instructions per
// hidden element).
//
// Matrix instruction layouts (32x32x16: lane (n, kb) of 32 x 2 holds 8 consecutive-k values of row /
// column n of its operand; register j of the result is row 8 (j / 4) + 4 kb + j % 4, column n).  The
// order of the k-values is free as long as both operands share it, which is used throughout: the result
// of the first product, packed in pairs of registers, IS an operand over the hidden channels of the next
// one, with k-step s, element e <-> hidden channel 16 s + 8 (e / 4) + 4 kb + e % 4 of the tile.  Nothing
// moves between lanes for it.  As in ndc_pwgemm.h a tile's 64 voxels are two matrix tiles, the even and
// the odd voxels, so that a lane holds both halves of an output word.
//
// Device code only; float32 accumulation, h and gu rounded to bf16 once, as the operands of the products
// they enter.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ndc_common.h"
#include "ndc_epilogue.h"
#include "ndc_mlp_host.h"
#include "ndc_pwgemm.h"

namespace ndc {
namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Params {
    const uint16_t *x, *gy, *res;   // (B, C, n)
    const float *stats;             // NORM: (mean, 1 / deviation) of each row of x
    const void *w1, *w2;
    const float *b1, *b2;           // 4C and C values, or null
    uint16_t *y;                    // forward: y; backward: gx
    float *part;                    // backward: part_floats(C) per workgroup
    long long n;                    // voxels per sample, a multiple of 64
    int tiles, tiles_per_sample;
};

__device__ inline float lo_bf16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ inline float hi_bf16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ inline bf16x8 frag(const u32x4 &v) { return __builtin_bit_cast(bf16x8, v); }
__device__ inline f32x16 mfma32(const bf16x8 &a, const bf16x8 &b, const f32x16 &c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The normal distribution's cdf, and exp(-u^2 / 2): erf by Abramowitz & Stegun 7.1.26, as in
// epilogue::act_fwd, with the scale of u folded into the constants.
__device__ inline float normal_cdf(float u, float &gauss)
{
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_fabsf(u), 0.23164189f, 1.f));
    gauss = __builtin_amdgcn_exp2f((u * -0.72134752f) * u);
    const float poly =
        t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
    const float erf = __builtin_copysignf(__builtin_fmaf(-poly, gauss, 1.f), u);
    return __builtin_fmaf(erf, 0.5f, 0.5f);
}

// The 8 values of a weight matrix a lane holds of one fragment, value e at at(e)
template <typename TW, class At> __device__ inline u32x4 weight_frag(const TW *w, At at)
{
    u32x4 r;
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) r[pr] = pack_bf16x2(Elem<TW>::load(w + at(2 * pr)), Elem<TW>::load(w + at(2 * pr + 1)));
    return r;
}
// element e of half kb <-> offset inside a 16-wide k-step, for operands that come out of a product
__device__ inline int result_k(int e, int kb) { return 8 * (e >> 2) + 4 * kb + (e & 3); }

// (even voxels, odd voxels) of 8 channel words
__device__ inline void split_words(const uint32_t (&raw)[8], u32x4 &even, u32x4 &odd)
{
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) {
        even[pr] = __builtin_amdgcn_perm(raw[2 * pr + 1], raw[2 * pr], 0x05040100u);
        odd[pr] = __builtin_amdgcn_perm(raw[2 * pr + 1], raw[2 * pr], 0x07060302u);
    }
}
__device__ inline const uint32_t *words(const uint16_t *p) { return reinterpret_cast<const uint32_t *>(p); }
__device__ inline uint32_t *words(uint16_t *p) { return reinterpret_cast<uint32_t *>(p); }

// ------------------------------------------------------------------ forward

// One wavefront takes 64 voxels and walks the hidden channels 32 at a time: product, GELU, rounded
// pairs, and on to the C / 32 output tiles it keeps.  Both weights sit in LDS in fragment order (64 KB at
// C = 64), packed by the workgroup itself from the float32 matrices (twice 64 KB that the L2 holds;
// a packing launch each costs more).  Workgroups are persistent, twelve wavefronts at C = 64: three per
// SIMD is what the 168 registers of a wavefront leave.
// NORM: x is normalised as it is loaded, and the residual is the x before that.
// HALF: a wavefront takes the even or the odd voxels of a tile, and a launch has twice as many: for few tiles,
// whose time is the GELUs of one wavefront one after the other (see forward_launch).
template <int C, typename TW, bool RES, int THREADS, bool NORM, bool HALF>
__global__ void __launch_bounds__(THREADS) forward_kernel(Params p)
{
    constexpr int H = 4 * C, S = C / 16, HT = H / 32, OT = C / 32, WAVES = THREADS / 64;
    __shared__ __attribute__((aligned(16))) u32x4 w1l[HT * S * 64];
    __shared__ __attribute__((aligned(16))) u32x4 w2l[HT * 2 * OT * 64];
    __shared__ __attribute__((aligned(16))) float b1l[H], b2l[C];
    for (int i = threadIdx.x; i < HT * S * 64; i += THREADS) {
        const int l = i & 63, f = i >> 6, s = f % S, ct = f / S;
        w1l[i] = weight_frag((const TW *)p.w1, [&](int e) { return (32 * ct + (l & 31)) * C + 16 * s + 8 * (l >> 5) + e; });
    }
    for (int i = threadIdx.x; i < HT * 2 * OT * 64; i += THREADS) {
        const int l = i & 63, f = i >> 6, o = f % OT, s = f / OT % 2, ct = f / (2 * OT);
        w2l[i] = weight_frag((const TW *)p.w2, [&](int e) {
            return (32 * o + (l & 31)) * H + 32 * ct + 16 * s + result_k(e, l >> 5);
        });
    }
    for (int i = threadIdx.x; i < H; i += THREADS) b1l[i] = p.b1 ? p.b1[i] : 0.f;
    for (int i = threadIdx.x; i < C; i += THREADS) b2l[i] = p.b2 ? p.b2[i] : 0.f;
    __syncthreads();

    const int lane = threadIdx.x & 63, n32 = lane & 31, kb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t xw = (uint32_t)(4 * kb) * (uint32_t)p.n + n32, yw = (uint32_t)(2 * kb) * (uint32_t)p.n + n32;
    constexpr int PER = HALF ? 2 : 1, NP = 2 / PER;   // wavefronts to a tile, parities to a wavefront
    const int nwaves = (int)gridDim.x * WAVES / PER, odd = wave % PER;
    for (int tile = ((int)blockIdx.x * WAVES + wave) / PER; tile < p.tiles; tile += nwaves) {
        const int b = __builtin_amdgcn_readfirstlane(tile / p.tiles_per_sample);
        const long long at0 = (long long)b * C * p.n + (long long)(tile - b * p.tiles_per_sample) * kTileVoxels;
        u32x4 xf[S][NP];
        {
            uint32_t raw[S][8];
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) raw[s][e] = words(p.x + at0 + (long long)(16 * s + e) * p.n)[xw];
            if constexpr (NORM) pwgemm::normalise_words<S>(raw, p.stats + 2 * (long long)b * C, kb);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                u32x4 even_odd[2];
                split_words(raw[s], even_odd[0], even_odd[1]);
                if constexpr (HALF) xf[s][0] = odd ? even_odd[1] : even_odd[0];
                else xf[s][0] = even_odd[0], xf[s][1] = even_odd[1];
            }
        }
        f32x16 acc[OT][NP];
#pragma unroll
        for (int o = 0; o < OT; ++o)
#pragma unroll
            for (int par = 0; par < NP; ++par) acc[o][par] = f32x16{};
#pragma unroll 1
        for (int ct = 0; ct < HT; ++ct) {
            // (the even and the odd voxels one after the other: side by side they spill registers)
#pragma unroll
            for (int par = 0; par < NP; ++par) {
                __builtin_amdgcn_sched_barrier(0);
                f32x16 u = {};
#pragma unroll
                for (int s = 0; s < S; ++s) u = mfma32(frag(w1l[(ct * S + s) * 64 + lane]), frag(xf[s][par]), u);
                u32x4 h[2];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 t4 = *reinterpret_cast<const float4 *>(b1l + 32 * ct + 8 * q + 4 * kb);
                    const float bq[4] = {t4.x, t4.y, t4.z, t4.w};
                    float a[4], unused;
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj) {
                        const float v = u[4 * q + jj] + bq[jj];
                        a[jj] = v * normal_cdf(v, unused);
                    }
                    h[q / 2][2 * (q & 1)] = pack_bf16x2(a[0], a[1]);
                    h[q / 2][2 * (q & 1) + 1] = pack_bf16x2(a[2], a[3]);
                }
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int o = 0; o < OT; ++o)
                        acc[o][par] = mfma32(frag(w2l[((ct * 2 + s) * OT + o) * 64 + lane]), frag(h[s]), acc[o][par]);
            }
        }
#pragma unroll
        for (int o = 0; o < OT; ++o) {
            uint32_t rw[16];
            if constexpr (RES) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    rw[j] = words(p.res + at0 + (long long)(32 * o + 8 * (j / 4) + j % 4) * p.n)[yw];
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float bj = b2l[32 * o + 8 * (j / 4) + 4 * kb + j % 4];
                uint32_t *to = words(p.y + at0 + (long long)(32 * o + 8 * (j / 4) + j % 4) * p.n) + yw;
                float y0 = acc[o][0][j] + bj, y1 = HALF ? 0.f : acc[o][NP - 1][j] + bj;
                if constexpr (HALF) {
                    if constexpr (RES) y0 += odd ? hi_bf16(rw[j]) : lo_bf16(rw[j]);
                    reinterpret_cast<uint16_t *>(to)[odd] = (uint16_t)pack_bf16x2(y0, 0.f);
                } else {
                    if constexpr (RES) y0 += lo_bf16(rw[j]), y1 += hi_bf16(rw[j]);
                    *to = pack_bf16x2(y0, y1);
                }
            }
        }
    }
}

// ------------------------------------------------------------------ backward

// A workgroup of C / 8 wavefronts takes 64 voxels at a time, wavefront w the hidden channels 32 w ..
// 32 w + 31 of them, with its slices of the weights in registers and the 32 x C tiles of gW1 and gW2 it
// owns accumulated there over the whole launch.  Per tile:
//   * the operands of all products over x and gy are made once per workgroup, in LDS in fragment order:
//     `col` fragments (lane <-> voxel, elements <-> 8 channels) and `row` fragments (lane <-> channel,
//     elements <-> 8 voxels); every wavefront makes one of each kind, from words requested a tile ahead;
//   * u and W2^T gy by matrix instructions, then gelu, gelu' and the rounding of h and gu;
//   * gu goes to LDS as operand fragments; behind the barrier every wavefront makes 16 rows of gx from
//     all hidden channels' (16x16x32 instructions, its slice of W1^T in registers);
//   * the weight gradients contract over voxels, i.e. want h and gu with the voxels inside a lane.  The
//     transposition is a product with the identity (exact): its result, packed, is that operand.
// Two barriers a tile.  The sums a workgroup ends with go to its row of `part`; the caller adds the rows
// in a fixed order.
// GX, G1, G2: x's gradient, the first projection's, the second's.  What none of them needs is not compiled in
// (gx may be null with GX, and is not stored then).
template <int C, typename TW, bool GX, bool G1, bool G2>
__global__ void __launch_bounds__(8 * C, 2) backward_kernel(Params p)
{
    constexpr bool GU = GX || G1;   // the hidden tensor's gradient is formed
    constexpr int H = 4 * C, S = C / 16, WAVES = C / 8, RB = C / 32;
    __shared__ __attribute__((aligned(16))) u32x4 col[2][S][2][64];        // [x, gy][k-step][parity]
    __shared__ __attribute__((aligned(16))) u32x4 row[2][RB][2][2][64];    // [x, gy][32 channels][k-step][parity]
    __shared__ __attribute__((aligned(16))) u32x4 gul[2 * WAVES][2][64];   // [hidden k-step][parity]
    __shared__ __attribute__((aligned(16))) u32x4 w1t[RB * 2][WAVES][64];  // [16 rows of W1^T][32 hidden channels]
    __shared__ __attribute__((aligned(16))) float b1l[H];
    const int lane = threadIdx.x & 63, n32 = lane & 31, kb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h0 = 32 * wave;   // this wavefront's hidden channels

    // weight slices: rows of W1 and of W2^T
    u32x4 w1f[S], w2f[S];
    const int n16 = lane & 15, kg = lane >> 4;
    const int gx_row = 16 * (wave >> 1), gx_half = wave & 1;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        w1f[s] = weight_frag((const TW *)p.w1, [&](int e) { return (h0 + n32) * C + 16 * s + 8 * kb + e; });
        if constexpr (GU) w2f[s] = weight_frag((const TW *)p.w2, [&](int e) { return (16 * s + 8 * kb + e) * H + h0 + n32; });
    }
    for (int i = threadIdx.x; GX && i < RB * 2 * WAVES * 64; i += 64 * WAVES) {
        const int l = i & 63, t = (i >> 6) % WAVES, r = (i >> 6) / WAVES, g = l >> 4;
        w1t[r][t][l] = weight_frag((const TW *)p.w1, [&](int e) {
            return (32 * t + 16 * (g >> 1) + result_k(e, g & 1)) * C + 16 * r + (l & 15);
        });
    }
    for (int i = threadIdx.x; i < H; i += 64 * WAVES) b1l[i] = p.b1 ? p.b1[i] : 0.f;
    // the identity as the second operand of a transposition
    u32x4 ident[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int pr = 0; pr < 4; ++pr)
            ident[s][pr] = (16 * s + result_k(2 * pr, kb) == n32 ? 0x3f80u : 0u) |
                           (16 * s + result_k(2 * pr + 1, kb) == n32 ? 0x3f800000u : 0u);

    f32x16 gw1[RB], gw2[RB];
    float gb1[16], gb2 = 0.f;
#pragma unroll
    for (int i = 0; i < RB; ++i) gw1[i] = f32x16{}, gw2[i] = f32x16{};
#pragma unroll
    for (int j = 0; j < 16; ++j) gb1[j] = 0.f;

    // what this wavefront stages: wavefronts below half of them x, the others gy
    const int second = wave >= WAVES / 2, unit = second ? wave - WAVES / 2 : wave;
    const int rb = unit >> 1, rs = unit & 1;
    const uint16_t *src = second ? p.gy : p.x;
    uint32_t cw[8];
    u32x4 rw[2];
    const bool wants_row = second ? G2 : G1, wants_col = !second || GU;
    auto request = [&](int tile) {
        const int b = __builtin_amdgcn_readfirstlane(tile / p.tiles_per_sample);
        const uint16_t *t0 = src + (long long)b * C * p.n + (long long)(tile - b * p.tiles_per_sample) * kTileVoxels;
        if (wants_col)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                cw[e] = words(t0 + (long long)(16 * unit + e) * p.n)[(uint32_t)(4 * kb) * (uint32_t)p.n + n32];
        if (!wants_row) return;
        const uint32_t lo = (uint32_t)n32 * (uint32_t)p.n + 8 * kb;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            rw[i] = *reinterpret_cast<const u32x4 *>(t0 + (long long)(32 * rb) * p.n + 16 * (2 * rs + i) + lo);
    };
    auto stage = [&]() {
        u32x4 even, odd;
        if (wants_col) {
            split_words(cw, even, odd);
            col[second][unit][0][lane] = even;
            col[second][unit][1][lane] = odd;
        }
        if (!wants_row) return;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                even[2 * i + k] = __builtin_amdgcn_perm(rw[i][2 * k + 1], rw[i][2 * k], 0x05040100u);
                odd[2 * i + k] = __builtin_amdgcn_perm(rw[i][2 * k + 1], rw[i][2 * k], 0x07060302u);
            }
        row[second][rb][rs][0][lane] = even;
        row[second][rb][rs][1][lane] = odd;
        if (second) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k) gb2 = dot2_bf16(rw[i][k], 0x3f803f80u, gb2);
        }
    };

    int tile = (int)blockIdx.x;
    if (tile < p.tiles) {
        request(tile);
        stage();
    }
    for (; tile < p.tiles; tile += (int)gridDim.x) {
        const int next = tile + (int)gridDim.x;
        __syncthreads();   // the fragments are there; the last tile's gu has been read
        if (next < p.tiles) request(next);
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            f32x16 u = {}, gh = {};
#pragma unroll
            for (int s = 0; s < S; ++s) {
                u = mfma32(frag(w1f[s]), frag(col[0][s][par][lane]), u);
                if constexpr (GU) gh = mfma32(frag(w2f[s]), frag(col[1][s][par][lane]), gh);
            }
            u32x4 hf[2], gf[2];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 t4 = *reinterpret_cast<const float4 *>(b1l + h0 + 8 * q + 4 * kb);
                const float bq[4] = {t4.x, t4.y, t4.z, t4.w};
                float h[4], g[4];
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const int j = 4 * q + jj;
                    float gauss;
                    const float v = u[j] + bq[jj], cdf = normal_cdf(v, gauss);
                    h[jj] = v * cdf;
                    g[jj] = gh[j] * __builtin_fmaf(v * 0.3989422804014327f, gauss, cdf);
                    if constexpr (G1) gb1[j] += g[jj];
                }
                hf[q / 2][2 * (q & 1)] = pack_bf16x2(h[0], h[1]);
                hf[q / 2][2 * (q & 1) + 1] = pack_bf16x2(h[2], h[3]);
                gf[q / 2][2 * (q & 1)] = pack_bf16x2(g[0], g[1]);
                gf[q / 2][2 * (q & 1) + 1] = pack_bf16x2(g[2], g[3]);
            }
            if constexpr (GX)
#pragma unroll
                for (int s = 0; s < 2; ++s) gul[2 * wave + s][par][lane] = gf[s];
            // voxels inside the lane, hidden channels along the lanes
            f32x16 ht = {}, gt = {};
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if constexpr (G2) ht = mfma32(frag(hf[s]), frag(ident[s]), ht);
                if constexpr (G1) gt = mfma32(frag(gf[s]), frag(ident[s]), gt);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                u32x4 hv, gv;
#pragma unroll
                for (int pr = 0; pr < 4; ++pr) {
                    hv[pr] = pack_bf16x2(ht[8 * s + 2 * pr], ht[8 * s + 2 * pr + 1]);
                    gv[pr] = pack_bf16x2(gt[8 * s + 2 * pr], gt[8 * s + 2 * pr + 1]);
                }
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    if constexpr (G1) gw1[i] = mfma32(frag(gv), frag(row[0][i][s][par][lane]), gw1[i]);   // hidden x input channel
                    if constexpr (G2) gw2[i] = mfma32(frag(row[1][i][s][par][lane]), frag(hv), gw2[i]);   // output channel x hidden
                }
            }
        }
        __syncthreads();   // gu of all hidden channels is there; the fragments have been read
        if (next < p.tiles) stage();
        if (!GX || !p.y) continue;
        f32x4 g0 = {}, g1 = {};
#pragma unroll
        for (int t = 0; t < WAVES; ++t) {
            const int ks = 2 * t + (kg >> 1), at = 16 * gx_half + n16 + 32 * (kg & 1);
            const bf16x8 a = frag(w1t[wave >> 1][t][lane]);
            g0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, frag(gul[ks][0][at]), g0, 0, 0, 0);
            g1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, frag(gul[ks][1][at]), g1, 0, 0, 0);
        }
        const int b = __builtin_amdgcn_readfirstlane(tile / p.tiles_per_sample);
        uint16_t *t0 = p.y + (long long)b * C * p.n + (long long)(tile - b * p.tiles_per_sample) * kTileVoxels;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            words(t0 + (long long)(gx_row + j) * p.n)[(uint32_t)(2 * kg) * (uint32_t)p.n + 16 * gx_half + n16] =
                pack_bf16x2(g0[j], g1[j]);
    }

    if constexpr (!G1 && !G2) return;
    float *o1 = p.part + (long long)blockIdx.x * part_floats(C), *o2 = o1 + H * C, *ob1 = o2 + H * C, *ob2 = ob1 + H;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int r = 8 * (j / 4) + 4 * kb + j % 4;
            if constexpr (G1) o1[(h0 + r) * C + 32 * i + n32] = gw1[i][j];
            if constexpr (G2) o2[(32 * i + r) * H + h0 + n32] = gw2[i][j];
        }
    if constexpr (G1)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float t = epilogue::half_sum(gb1[j]);
            if (n32 == 31) ob1[h0 + 8 * (j / 4) + 4 * kb + j % 4] = t;
        }
    if (G2 && second) ob2[(2 * rs + kb) * C + 32 * rb + n32] = gb2;
}

// The workgroups' partial results added up: thread (quad, j) of 32 x 8 takes four neighbouring values
// of the parts j, j + 8, ... in order, eight parts in flight, then the eight sums in order.  (One value a
// thread, strided_sum_kernel, took 16.5 us for the 34 MB of C = 64.)  Results that are null are not added up.
template <int C>
__global__ void __launch_bounds__(256) sum_kernel(const float *part, int nparts, float *gw1, float *gb1, float *gw2, float *gb2)
{
    constexpr int H = 4 * C, NW = H * C, first = 2 * NW + H;   // from `first` on: four rows of gb2
    constexpr long long stride = part_floats(C);
    __shared__ f32x4 buf[8][32];
    const int qx = threadIdx.x & 31, j = threadIdx.x >> 5;
    const int o = (int)(blockIdx.x * 32 + qx) * 4;
    float *const base = o < NW ? gw1 : o < 2 * NW ? gw2 : o < first ? gb1 : o < first + C ? gb2 : nullptr;
    f32x4 acc = {};
    if (base && o < first) {
        const float *at = part + o;
        int k = j;
        for (; k + 56 < nparts; k += 64) {
            f32x4 t[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) t[i] = *reinterpret_cast<const f32x4 *>(at + (k + 8 * i) * stride);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc += t[i];
        }
        for (; k < nparts; k += 8) acc += *reinterpret_cast<const f32x4 *>(at + k * stride);
    } else if (base) {
        for (int k = j; k < nparts; k += 8) {
            const float *at = part + o + k * stride;
            f32x4 t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] = *reinterpret_cast<const f32x4 *>(at + i * C);
            acc += (t[0] + t[1]) + (t[2] + t[3]);
        }
    }
    buf[j][qx] = acc;
    __syncthreads();
    if (j == 0 && base) {
        f32x4 v = buf[0][qx];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += buf[i][qx];
        float *out = base + (o < NW ? o : o < 2 * NW ? o - NW : o < first ? o - 2 * NW : o - first);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = v[i];
    }
}

}  // namespace mlp
}  // namespace ndc
