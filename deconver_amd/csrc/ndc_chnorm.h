// Normalisation over the CHANNEL axis of a channel-first tensor (B, C, n): for every voxel,
//   y[b][c][i] = (x[b][c][i] - mean[b][i]) * rstd[b][i] * weight[c] + bias[c]
// with mean and (biased) variance taken over c.  This is the reference's LayerNorm
// (deconver/layers/norm.py:25-34: nn.LayerNorm applied with the channel axis moved last) on the
// layout the tensors already have: lanes run along the voxels (16 bytes each), a loop runs over
// the channels, so every access is a contiguous run and nothing is transposed.
//
// Up to 256 channels (held_*): a workgroup's eight wavefronts each take every eighth channel of the
// same 64 lanes of voxels (two a lane where the rows allow it) and hold them in registers, so the
// tensors are read once; a wavefront's own mean and squared deviations per voxel are merged through
// LDS.  One thread per voxel over all channels, which this replaces there, read its tensors twice,
// ran one dependent load after another and left most of the chip idle on grids of 10^5 voxels.
//   forward : mean and squared deviations of the slices, merged; y.  stats[b][0][i] = mean,
//             stats[b][1][i] = rstd.
//   backward: sums of g w and g w xhat per voxel, merged;
//             gx = rstd (g w - mean_c(g w) - xhat mean_c(g w xhat));
//             the sums over voxels of g xhat and g stay in registers over the voxels a workgroup
//             walks and become one row of `partial` (the affine gradients are the rows' sums).
// HBM traffic: forward 1 read + 1 write of the tensor, backward 2 reads + 1 write.  64 channels x
// 137 280 voxels in bfloat16: 15 and 24 us (35 and 53 MB); as float32 between conversions, a thread a
// voxel, 44 and 74 us and four conversions of 10 us.
// More channels (forward_kernel, backward_kernel): a thread per voxel (16 bytes of them) and two
// loops over the channels, 2 reads + 1 write and 4 reads + 1 write, one row per wavefront.
// float32 arithmetic.  Device code only.
#pragma once
#include "ndc_exec.h"
#include "ndc_rownorm.h"

namespace ndc {
namespace chnorm {

using rownorm::kThreads;
using rownorm::Vec;

struct Shape {
    long long n;      // voxels per (sample, channel)
    int channels;
    int blocks;       // workgroups per sample
};

template <typename T, bool VEC> struct Lanes {
    static constexpr int N = VEC ? Vec<T>::N : 1;
    float v[N];
    __device__ void load(const T *p)
    {
        if constexpr (VEC) {
            const Vec<T> x = *reinterpret_cast<const Vec<T> *>(p);
#pragma unroll
            for (int e = 0; e < N; ++e) v[e] = x.get(e);
        } else {
            v[0] = Elem<T>::load(p);
        }
    }
    __device__ void store(T *p) const
    {
        if constexpr (VEC) {
            Vec<T> r;
            if constexpr (sizeof(T) == 2) {
#pragma unroll
                for (int q = 0; q < N / 2; ++q) r.set_pair(q, v[2 * q], v[2 * q + 1]);
            } else {
#pragma unroll
                for (int e = 0; e < N; ++e) r.set(e, v[e]);
            }
            *reinterpret_cast<Vec<T> *>(p) = r;
        } else {
            Elem<T>::store(p, v[0]);
        }
    }
};

// LV voxels of one channel as they lie in memory
template <typename T, int LV> struct Held;
template <> struct Held<bf16_t, 1> {
    bf16_t w;
    __device__ float get(int) const { return bf16_to_float(w); }
};
template <> struct Held<bf16_t, 2> {
    uint32_t w;
    __device__ float get(int e) const { return __uint_as_float(e ? w & 0xffff0000u : w << 16); }
};
template <> struct Held<float, 1> {
    float w;
    __device__ float get(int) const { return w; }
};
template <> struct Held<float, 2> {
    float2 w;
    __device__ float get(int e) const { return e ? w.y : w.x; }
};

static constexpr int kSlices = 8, kHeldThreads = 64 * kSlices, kHeldChannels = 256;

struct HeldShape {
    long long n;          // voxels per (sample, channel)
    int channels;
    int groups;           // workgroups per sample
    long long tiles;      // runs of 64 * LV voxels per sample
    long long parts;      // rows of `partial`: those past the workgroups are set to zero
};

template <typename T, int LV, int CPT>
__global__ void __launch_bounds__(kHeldThreads)
held_forward_kernel(const T *x, const float *weight, const float *bias, T *y, float *stats, HeldShape s, float eps)
{
    typedef Held<T, LV> H;
    __shared__ float buf[2][kSlices][2][64 * LV];
    const int lane = threadIdx.x & 63, slice = uniform_int((int)threadIdx.x >> 6);
    const long long b = blockIdx.x / s.groups;
    const T *xs = x + b * s.channels * s.n;
    T *ys = y + b * s.channels * s.n;
    const float own = (float)((s.channels - slice + kSlices - 1) / kSlices), inv_own = own > 0.f ? 1.f / own : 0.f;
    const float inv_c = 1.f / (float)s.channels;
    int parity = 0;
    for (long long tile = blockIdx.x % s.groups; tile < s.tiles; tile += s.groups, parity ^= 1) {
        const long long i = (tile * 64 + lane) * LV;
        const bool in = i < s.n;
        const long long at = in ? i : 0;
        H h[CPT];
#pragma unroll
        for (int k = 0; k < CPT; ++k)
            if (slice + k * kSlices < s.channels)
                h[k] = *reinterpret_cast<const H *>(xs + (slice + k * kSlices) * s.n + at);
        float m[LV], q[LV];
#pragma unroll
        for (int e = 0; e < LV; ++e) m[e] = q[e] = 0.f;
#pragma unroll
        for (int k = 0; k < CPT; ++k)
            if (slice + k * kSlices < s.channels)
#pragma unroll
                for (int e = 0; e < LV; ++e) m[e] += h[k].get(e);
#pragma unroll
        for (int e = 0; e < LV; ++e) m[e] *= inv_own;
#pragma unroll
        for (int k = 0; k < CPT; ++k)
            if (slice + k * kSlices < s.channels)
#pragma unroll
                for (int e = 0; e < LV; ++e) {
                    const float d = h[k].get(e) - m[e];
                    q[e] += d * d;
                }
#pragma unroll
        for (int e = 0; e < LV; ++e) {
            buf[parity][slice][0][e * 64 + lane] = m[e];
            buf[parity][slice][1][e * 64 + lane] = q[e];
        }
        __syncthreads();   // (the other half is written next: no second barrier)
        float mean[LV], rstd[LV];
#pragma unroll
        for (int e = 0; e < LV; ++e) {
            // the slices' means and deviations merged: no cancellation whatever the values' offset
            float pm[kSlices], sum = 0.f, m2 = 0.f;
#pragma unroll
            for (int j = 0; j < kSlices; ++j) {
                pm[j] = buf[parity][j][0][e * 64 + lane];
                sum += pm[j] * (float)((s.channels - j + kSlices - 1) / kSlices);
            }
            mean[e] = sum * inv_c;
#pragma unroll
            for (int j = 0; j < kSlices; ++j) {
                const float d = pm[j] - mean[e];
                m2 += buf[parity][j][1][e * 64 + lane] + d * d * (float)((s.channels - j + kSlices - 1) / kSlices);
            }
            rstd[e] = 1.f / sqrtf(m2 * inv_c + eps);
        }
        if (!in) continue;
        if (slice == 0) {
#pragma unroll
            for (int e = 0; e < LV; ++e) {
                stats[(b * 2 + 0) * s.n + i + e] = mean[e];
                stats[(b * 2 + 1) * s.n + i + e] = rstd[e];
            }
        }
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int c = slice + k * kSlices;
            if (c >= s.channels) continue;
            const float w = weight ? weight[c] : 1.f, bb = bias ? bias[c] : 0.f;
            float v[LV];
#pragma unroll
            for (int e = 0; e < LV; ++e) v[e] = (h[k].get(e) - mean[e]) * rstd[e] * w + bb;
            VecIO<T, LV>::store(ys + c * s.n + i, v);
        }
    }
}

// partial: (parts, channels, 2) floats, or null
template <typename T, int LV, int CPT>
__global__ void __launch_bounds__(kHeldThreads)
held_backward_kernel(const T *gy, const T *x, const float *stats, const float *weight, T *gx, float *partial, HeldShape s)
{
    typedef Held<T, LV> H;
    __shared__ float buf[2][kSlices][2][64 * LV];
    const int lane = threadIdx.x & 63, slice = uniform_int((int)threadIdx.x >> 6);
    const long long b = blockIdx.x / s.groups;
    const T *xs = x + b * s.channels * s.n, *gs = gy + b * s.channels * s.n;
    T *os = gx + b * s.channels * s.n;
    const float inv_c = 1.f / (float)s.channels;
    float pw[CPT], pb[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) pw[k] = pb[k] = 0.f;
    int parity = 0;
    for (long long tile = blockIdx.x % s.groups; tile < s.tiles; tile += s.groups, parity ^= 1) {
        const long long i = (tile * 64 + lane) * LV;
        const bool in = i < s.n;
        const long long at = in ? i : 0;
        H hx[CPT], hg[CPT];
#pragma unroll
        for (int k = 0; k < CPT; ++k)
            if (slice + k * kSlices < s.channels) {
                hx[k] = *reinterpret_cast<const H *>(xs + (slice + k * kSlices) * s.n + at);
                hg[k] = *reinterpret_cast<const H *>(gs + (slice + k * kSlices) * s.n + at);
            }
        float mean[LV], rstd[LV], s1[LV], s2[LV];
#pragma unroll
        for (int e = 0; e < LV; ++e) {
            mean[e] = stats[(b * 2 + 0) * s.n + at + e];
            rstd[e] = stats[(b * 2 + 1) * s.n + at + e];
            s1[e] = s2[e] = 0.f;
        }
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int c = slice + k * kSlices;
            if (c >= s.channels) continue;
            const float w = weight ? weight[c] : 1.f;
#pragma unroll
            for (int e = 0; e < LV; ++e) {
                const float g = hg[k].get(e), xh = (hx[k].get(e) - mean[e]) * rstd[e];
                s1[e] += g * w;
                s2[e] += g * w * xh;
                pw[k] += in ? g * xh : 0.f;
                pb[k] += in ? g : 0.f;
            }
        }
#pragma unroll
        for (int e = 0; e < LV; ++e) {
            buf[parity][slice][0][e * 64 + lane] = s1[e];
            buf[parity][slice][1][e * 64 + lane] = s2[e];
        }
        __syncthreads();   // (the other half is written next: no second barrier)
#pragma unroll
        for (int e = 0; e < LV; ++e) {
            s1[e] = s2[e] = 0.f;
#pragma unroll
            for (int j = 0; j < kSlices; ++j) {
                s1[e] += buf[parity][j][0][e * 64 + lane];
                s2[e] += buf[parity][j][1][e * 64 + lane];
            }
        }
        if (!in) continue;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            const int c = slice + k * kSlices;
            if (c >= s.channels) continue;
            const float w = weight ? weight[c] : 1.f;
            float v[LV];
#pragma unroll
            for (int e = 0; e < LV; ++e) {
                const float xh = (hx[k].get(e) - mean[e]) * rstd[e];
                v[e] = rstd[e] * (hg[k].get(e) * w - s1[e] * inv_c - xh * s2[e] * inv_c);
            }
            VecIO<T, LV>::store(os + c * s.n + i, v);
        }
    }
    if (!partial) return;
    struct None {};
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        const int c = slice + k * kSlices;
        if (c >= s.channels) continue;
        const float w = DeviceExec<None>::wave_sum(pw[k]), g = DeviceExec<None>::wave_sum(pb[k]);
        if (lane == 63) {
            partial[((long long)blockIdx.x * s.channels + c) * 2] = w;
            partial[((long long)blockIdx.x * s.channels + c) * 2 + 1] = g;
        }
    }
    for (long long r = (long long)blockIdx.x + gridDim.x; r < s.parts; r += gridDim.x)
        for (int c = threadIdx.x; c < 2 * s.channels; c += kHeldThreads) partial[r * s.channels * 2 + c] = 0.f;
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
forward_kernel(const T *x, const float *weight, const float *bias, T *y, float *stats, Shape s, float eps)
{
    typedef Lanes<T, VEC> L;
    const long long b = blockIdx.x / s.blocks;
    const long long i = ((long long)(blockIdx.x % s.blocks) * kThreads + threadIdx.x) * L::N;
    if (i >= s.n) return;
    const T *xb = x + b * s.channels * s.n + i;
    T *yb = y + b * s.channels * s.n + i;
    L t;
    // running mean and squared deviations per voxel (Welford): no cancellation whatever the
    // offset of the values
    float mean[L::N], m2[L::N];
#pragma unroll
    for (int e = 0; e < L::N; ++e) mean[e] = m2[e] = 0.f;
    for (int c = 0; c < s.channels; ++c) {
        t.load(xb + c * s.n);
        const float rk = 1.f / (float)(c + 1);
#pragma unroll
        for (int e = 0; e < L::N; ++e) {
            const float d = t.v[e] - mean[e];
            mean[e] += d * rk;
            m2[e] += d * (t.v[e] - mean[e]);
        }
    }
    const float inv_c = 1.f / (float)s.channels;
    float rstd[L::N];
#pragma unroll
    for (int e = 0; e < L::N; ++e) {
        rstd[e] = 1.f / sqrtf(m2[e] * inv_c + eps);
        stats[(b * 2 + 0) * s.n + i + e] = mean[e];
        stats[(b * 2 + 1) * s.n + i + e] = rstd[e];
    }
    for (int c = 0; c < s.channels; ++c) {
        const float w = weight ? weight[c] : 1.f, bb = bias ? bias[c] : 0.f;
        t.load(xb + c * s.n);
#pragma unroll
        for (int e = 0; e < L::N; ++e) t.v[e] = (t.v[e] - mean[e]) * rstd[e] * w + bb;
        t.store(yb + c * s.n);
    }
}

// partial: (gridDim.x * wavefronts per workgroup, channels, 2) floats, or null
template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
backward_kernel(const T *gy, const T *x, const float *stats, const float *weight, T *gx, float *partial,
                Shape s)
{
    typedef Lanes<T, VEC> L;
    const long long b = blockIdx.x / s.blocks;
    const long long i = ((long long)(blockIdx.x % s.blocks) * kThreads + threadIdx.x) * L::N;
    const bool active = i < s.n;
    const long long at = active ? i : 0;   // idle lanes read voxel 0 and contribute zeros
    const T *gb = gy + b * s.channels * s.n + at, *xb = x + b * s.channels * s.n + at;
    T *ob = gx + b * s.channels * s.n + at;
    float mean[L::N], rstd[L::N], s1[L::N], s2[L::N];
#pragma unroll
    for (int e = 0; e < L::N; ++e) {
        mean[e] = stats[(b * 2 + 0) * s.n + at + e];
        rstd[e] = active ? stats[(b * 2 + 1) * s.n + at + e] : 0.f;
        s1[e] = s2[e] = 0.f;
    }
    float *mine = partial ? partial + ((long long)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)) * s.channels * 2
                          : nullptr;
    L g, t;
    for (int c = 0; c < s.channels; ++c) {
        const float w = weight ? weight[c] : 1.f;
        g.load(gb + c * s.n);
        t.load(xb + c * s.n);
        float pw = 0.f, pb = 0.f;
#pragma unroll
        for (int e = 0; e < L::N; ++e) {
            const float gv = active ? g.v[e] : 0.f;
            const float xh = (t.v[e] - mean[e]) * rstd[e];
            s1[e] += gv * w;
            s2[e] += gv * w * xh;
            pw += gv * xh;
            pb += gv;
        }
        if (mine) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                pw += __shfl_down(pw, off, 64);
                pb += __shfl_down(pb, off, 64);
            }
            if ((threadIdx.x & 63) == 0) {
                mine[2 * c] = pw;
                mine[2 * c + 1] = pb;
            }
        }
    }
    if (!active) return;
    const float inv_c = 1.f / (float)s.channels;
    for (int c = 0; c < s.channels; ++c) {
        const float w = weight ? weight[c] : 1.f;
        g.load(gb + c * s.n);
        t.load(xb + c * s.n);
#pragma unroll
        for (int e = 0; e < L::N; ++e) {
            const float xh = (t.v[e] - mean[e]) * rstd[e];
            t.v[e] = rstd[e] * (g.v[e] * w - s1[e] * inv_c - xh * s2[e] * inv_c);
        }
        t.store(ob + c * s.n);
    }
}

}  // namespace chnorm
}  // namespace ndc
