// AdamW over a list of float32 tensors (Loshchilov & Hutter, "Decoupled weight decay regularization"),
//
//   p <- p (1 - lr wd),  m <- m + (1 - b1) (g - m),  v <- b2 v + (1 - b2) g^2,
//   p <- p - lr / (1 - b1^t) * m / (sqrt(v) / sqrt(1 - b2^t) + eps),        t = *step + 1,
//
// the step counters (one float per tensor) on the device, so that a recorded step counts on.  Memory bound:
// 28 bytes a parameter.  The library's fused form deals 64 K elements to a workgroup, which leaves most of the
// chip idle for a network of this kind (some 140 tensors, 0.2 ms in four launches); here it is 4 K a workgroup,
// the tensors of a launch named in its arguments.  A recorded training step on one 128^2 image went from
// 2.17 to 2.07 ms by it.  Against float64 after twelve steps: parameters 9e-9 (the library's form 1.3e-8), first
// moments 5e-8, second 6e-8 (both as the library's; with all of it in float32 1.3e-7).
//
// Device code only.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/deconver_ndc.h"

namespace ndc {
namespace adamw {

static const int kTensors = 64, kSteps = 400;       // to a launch: what its 4 KB of arguments hold
static const int kThreads = 256, kChunk = 4096;     // elements of a workgroup

struct Params {
    ndc_adamw_tensor t[kTensors];
    uint32_t first[kTensors];       // a tensor's first workgroup
    int count;
    double beta1, beta2, lr, decay;   // decay: 1 - lr wd
    float eps;
};
struct Steps {
    float *step[kSteps];
    int count;
};

static __global__ void __launch_bounds__(kThreads) update_kernel(Params q)
{
    __shared__ float scale[2];
    int lo = 0, hi = q.count - 1;   // the last tensor that starts at or before this workgroup
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (q.first[mid] <= blockIdx.x) lo = mid; else hi = mid - 1;
    }
    const ndc_adamw_tensor t = q.t[lo];
    if (threadIdx.x == 0) {
        const double n = (double)*t.step + 1.0;
        scale[0] = (float)(q.lr / (1.0 - pow(q.beta1, n)));
        scale[1] = (float)sqrt(1.0 - pow(q.beta2, n));
    }
    __syncthreads();
    const float size = scale[0], root = scale[1];
    auto one = [&](float &p, float g, float &m, float &v) {
        // (factors next to one, times values kept for thousands of steps: rounded to float32 they are a bias)
        m = (float)(m + (1.0 - q.beta1) * ((double)g - m));
        v = (float)(q.beta2 * v + (1.0 - q.beta2) * ((double)g * g));
        p = (float)(p * q.decay - (double)size * (m / (sqrtf(v) / root + q.eps)));
    };
    const int64_t begin = (int64_t)(blockIdx.x - q.first[lo]) * kChunk;
    const int have = (int)(t.n - begin < kChunk ? t.n - begin : kChunk);
    float *p = t.param + begin, *m = t.m + begin, *v = t.v + begin;
    const float *g = t.grad + begin;
    int i = threadIdx.x;
    if ((((uintptr_t)p | (uintptr_t)g | (uintptr_t)m | (uintptr_t)v) & 15u) == 0) {
        for (; i < have / 4; i += kThreads) {
            float4 p4 = ((float4 *)p)[i], m4 = ((float4 *)m)[i], v4 = ((float4 *)v)[i];
            const float4 g4 = ((const float4 *)g)[i];
            one(p4.x, g4.x, m4.x, v4.x);
            one(p4.y, g4.y, m4.y, v4.y);
            one(p4.z, g4.z, m4.z, v4.z);
            one(p4.w, g4.w, m4.w, v4.w);
            ((float4 *)p)[i] = p4, ((float4 *)m)[i] = m4, ((float4 *)v)[i] = v4;
        }
        i = have / 4 * 4 + threadIdx.x;
    }
    for (; i < have; i += kThreads) one(p[i], g[i], m[i], v[i]);
}

// (behind the updates: their workgroups read the counters)
static __global__ void __launch_bounds__(64) count_kernel(Steps q)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i < q.count) *q.step[i] += 1.f;
}

}  // namespace adamw
}  // namespace ndc
