// Binary cross-entropy on logits plus soft Dice loss (+1 smoothing) over the rows (sample, channel) of a
// (B, C, *S) tensor,
//
//   loss = mean(max(l, 0) - l y + log(1 + exp(-|l|))) + mean_r(1 - (2 S_py + 1) / (S_p + S_y + 1)),
//   p = sigmoid(l),  S_py, S_p, S_y: sums over row r,
//
// and its gradient.  Out of tensor operations it is some 45 launches a training step, which is what small
// images and volumes spend a twelfth of their step on; here it is one pass that leaves four sums per part of
// a row, one workgroup that adds them (in a fixed order), and one pass for the gradient.  float32 arithmetic.
// The passes are bound by their launches at these sizes and by memory at large ones (8 bytes an element, then
// 12).  A captured training step on one 128^2 image went from 2.35 to 2.27 ms by it, an uncaptured one on a
// 32^3 volume, which the host paces, from 4.6 to 4.3 ms.
// Device code only.
#pragma once
#include <hip/hip_runtime.h>

namespace ndc {
namespace loss {

static const int kThreads = 256;
static const int kFinish = 1024;

__device__ inline float wave_total(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// partial[row][part] = (sum of the cross-entropy terms, S_py, S_p, S_y) of the part
static __global__ void __launch_bounds__(kThreads) sums_kernel(const float *l, const float *y, float4 *partial, long long n, int parts, long long chunk)
{
    __shared__ float buf[4][kThreads / 64];
    const long long row = blockIdx.x / parts;
    const int part = blockIdx.x % parts;
    const long long lo = part * chunk, hi = lo + chunk < n ? lo + chunk : n;
    const float *lr = l + row * n;
    const float *yr = y + row * n;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (long long i = lo + threadIdx.x; i < hi; i += kThreads) {
        const float v = lr[i], t = yr[i];
        const float e = expf(-fabsf(v)), p = (v >= 0.f ? 1.f : e) / (1.f + e);
        s[0] += (1.f - t) * v + (fmaxf(-v, 0.f) + log1pf(e));
        s[1] += p * t;
        s[2] += p;
        s[3] += t;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        s[k] = wave_total(s[k]);
        if ((threadIdx.x & 63) == 0) buf[k][threadIdx.x >> 6] = s[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float t[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = (buf[k][0] + buf[k][1]) + (buf[k][2] + buf[k][3]);
        partial[blockIdx.x] = make_float4(t[0], t[1], t[2], t[3]);
    }
}

// loss, and per row the coefficients of the gradient, coef[row] = ((2 S_py + 1) / (R D^2), 1 / (R D)),
// D = S_p + S_y + 1, R rows.  One workgroup in all; `width` = 2^log_width lanes a row, the first power of two that
// holds its parts, at most a wavefront.  (A wavefront a row whatever its parts: 1024 rows of one part each were 64
// trips to memory one after the other, 82 us for the loss of 64 x 16 rows of 64 and its gradient, 11 now; in tensor
// operations 76.)
static __global__ void __launch_bounds__(kFinish) finish_kernel(const float4 *partial, float2 *coef, float *loss, int rows, int parts,
                                                                  int log_width, float inv_total)
{
    __shared__ float buf[2][kFinish];
    const int width = 1 << log_width, lane = threadIdx.x & 63, first = threadIdx.x & (width - 1), group = threadIdx.x >> log_width;
    const int groups = kFinish >> log_width;
    const float inv_rows = 1.f / (float)rows;
    float bce = 0.f, dice = 0.f;
    // (all lanes of a wavefront take all trips: they exchange sums)
    for (int r0 = 0; r0 < rows; r0 += groups) {
        const int r = r0 + group;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        for (int q = first; q < parts && r < rows; q += width) {
            const float4 v = partial[(long long)r * parts + q];
            s[0] += v.x, s[1] += v.y, s[2] += v.z, s[3] += v.w;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
            if (off < width)
#pragma unroll
                for (int k = 0; k < 4; ++k) s[k] += __shfl_xor(s[k], off, 64);
        if (first == 0 && r < rows) {
            const float num = 2.f * s[1] + 1.f, den = s[2] + s[3] + 1.f;
            bce += s[0];
            dice += 1.f - num / den;
            coef[r] = make_float2(num / (den * den) * inv_rows, inv_rows / den);
        }
    }
    if (first == 0) buf[0][group] = bce, buf[1][group] = dice;
    __syncthreads();
    if (threadIdx.x < 64) {
        float b = 0.f, d = 0.f;
        for (int i = lane; i < groups; i += 64) b += buf[0][i], d += buf[1][i];
        b = wave_total(b), d = wave_total(d);
        if (lane == 0) *loss = b * inv_total + d * inv_rows;
    }
}

// gl = g ((p - y) / (R n) + p (1 - p) (coef.x - 2 y coef.y)), g read from the device
static __global__ void __launch_bounds__(kThreads) grad_kernel(const float *l, const float *y, const float2 *coef, const float *g, float *gl,
                                                        long long n, int parts, long long chunk, float inv_total)
{
    const long long row = blockIdx.x / parts;
    const int part = blockIdx.x % parts;
    const long long lo = part * chunk, hi = lo + chunk < n ? lo + chunk : n;
    const float2 c = coef[row];
    const float gv = *g;
#pragma unroll 4
    for (long long i = lo + threadIdx.x; i < hi; i += kThreads) {
        const float v = l[row * n + i], t = y[row * n + i];
        const float e = expf(-fabsf(v)), p = (v >= 0.f ? 1.f : e) / (1.f + e);
        gl[row * n + i] = gv * ((p - t) * inv_total + p * (1.f - p) * (c.x - 2.f * t * c.y));
    }
}

}  // namespace loss
}  // namespace ndc
