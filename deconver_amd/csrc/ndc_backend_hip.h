// Launch primitives of the HIP (gfx950) build: the `Backend` the shared host logic is written
// against.  Included by the translation units that instantiate kernels through it.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "ndc_common.h"
#include "ndc_exec.h"
#include "ndc_rownorm.h"
#include "ndc_epilogue.h"
#include "ndc_regroup.h"
#include "ndc_chnorm.h"
#include "ndc_pwgemm.h"
#include "ndc_gemm_host.h"
#include "ndc_mlp_host.h"
#include "ndc_loss.h"
#include "ndc_direct.h"
#include "ndc_adamw.h"

#define NDC_LAMBDA __host__ __device__

namespace ndc {

template <class F>
__global__ void __launch_bounds__(256) elementwise_kernel(long long n, F f)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += stride)
        f(idx);
}

// f(unit, position): the unit is the same for a whole workgroup, lanes run along the positions
template <class F>
__global__ void __launch_bounds__(128) per_unit_kernel(unsigned blocks, long long npos, F f)
{
    const unsigned u = blockIdx.x / blocks;
    const long long pos = (long long)(blockIdx.x - u * blocks) * 128 + threadIdx.x;
    if (pos < npos) f((int)u, pos);
}

// f.run(unit, position, weights): ... with the unit's weights in LDS
template <class F, bool STAGED>
__global__ void __launch_bounds__(128) weighted_unit_kernel(unsigned blocks, long long npos, F f)
{
    extern __shared__ __attribute__((aligned(16))) float weights[];
    const unsigned u = blockIdx.x / blocks;
    const long long pos = (long long)(blockIdx.x - u * blocks) * 128 + threadIdx.x;
    if constexpr (STAGED) {
        f.stage((int)u, weights, threadIdx.x, 128);
        __syncthreads();
    }
    if (pos < npos) f.template run<STAGED>((int)u, pos, weights);
}

// F::N sums over the threads of a workgroup, one workgroup per unit: f.sums gives a thread's
// own, f.put takes the totals
template <class F> __global__ void __launch_bounds__(256) unit_sums_kernel(F f)
{
    struct None {};
    __shared__ float lds[4 * F::N];
    const int u = (int)blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float acc[F::N];
    f.sums(u, tid, 256, acc);
#pragma unroll
    for (int i = 0; i < F::N; ++i) {
        const float v = DeviceExec<None>::wave_sum(acc[i]);
        if (lane == 63) lds[wave * F::N + i] = v;
    }
    __syncthreads();
    for (int i = tid; i < F::N; i += 256)
        f.put(u, i, ((lds[i] + lds[F::N + i]) + lds[2 * F::N + i]) + lds[3 * F::N + i]);
}

// put(o, sum over p < nparts of term(o, p)) for o < nout.  A workgroup sums 32 outputs:
// thread (o, j), j < 8, adds the terms p = j, j + 8, ... in order, then thread (o, 0) adds the
// eight partial sums in order -- a fixed association, so results are reproducible.  Threads
// with consecutive o are neighbours, so a `term` that is contiguous in o reads coalesced.
// What bounds it is the latency of a term's load, so eight of a thread's terms are requested
// before the first is added (the 256 x 64 weight gradient over 137 280 voxels, 512 terms a sum:
// 17 -> 6.7 us a launch).
template <class P, class F>
__global__ void __launch_bounds__(256) strided_sum_kernel(int nout, int nparts, P put, F term)
{
    __shared__ float buf[8][33];
    const int ox = threadIdx.x & 31, j = threadIdx.x >> 5;
    const int o = (int)blockIdx.x * 32 + ox;
    float acc = 0.f;
    if (o < nout) {
        int p = j;
        for (; p + 56 < nparts; p += 64) {
            float t[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) t[k] = term(o, p + 8 * k);
#pragma unroll
            for (int k = 0; k < 8; ++k) acc += t[k];
        }
        for (; p < nparts; p += 8) acc += term(o, p);
    }
    buf[j][ox] = acc;
    __syncthreads();
    if (j == 0 && o < nout) {
        float total = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) total += buf[k][ox];
        put(o, total);
    }
}

// Batched matrix transposition dst[b][k][r] = src[b][r][k] (R rows, K columns per batch entry)
// of 16-bit elements, two at a time: a workgroup moves a 64 x 64 tile through LDS, reading
// 32-bit words along K and writing 32-bit words along R (R, K even, both pointers 4-byte
// aligned).  The copy between the channels-last layout (B, S, C) and the channel-first layout
// (B, C, S) the update kernels read is this transposition with (R, K) = (S, C) or (C, S).
static __global__ void __launch_bounds__(256)
transpose_pairs_kernel(const uint32_t *src, uint32_t *dst, long long R, long long K, long long tiles_r,
                       long long tiles_k)
{
    __shared__ uint16_t tile[64][66];
    long long blk = blockIdx.x;
    const long long tk = blk % tiles_k;
    blk /= tiles_k;
    const long long tr = blk % tiles_r, b = blk / tiles_r;
    const long long row0 = tr * 64, col0 = tk * 64;
    const uint32_t *s = src + b * (R * K / 2);
    uint32_t *d = dst + b * (R * K / 2);
    const int w = threadIdx.x & 31, q = threadIdx.x >> 5;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const int r = q + 8 * it;
        uint32_t v = 0u;
        if (row0 + r < R && col0 + 2 * w < K) v = s[((row0 + r) * K + col0) / 2 + w];
        *reinterpret_cast<uint32_t *>(&tile[r][2 * w]) = v;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const int k = q + 8 * it;
        if (col0 + k < K && row0 + 2 * w < R)
            d[((col0 + k) * R + row0) / 2 + w] = (uint32_t)tile[2 * w][k] | ((uint32_t)tile[2 * w + 1][k] << 16);
    }
}

// The same for elements of ESZ bytes (2 or 4), one at a time: any R, K and alignment.
template <typename E>
__global__ void __launch_bounds__(256)
transpose_kernel(const E *src, E *dst, long long R, long long K, long long tiles_r, long long tiles_k)
{
    __shared__ E tile[32][33];
    long long blk = blockIdx.x;
    const long long tk = blk % tiles_k;
    blk /= tiles_k;
    const long long tr = blk % tiles_r, b = blk / tiles_r;
    const long long row0 = tr * 32, col0 = tk * 32;
    const E *s = src + b * R * K;
    E *d = dst + b * R * K;
    const int w = threadIdx.x & 31, q = threadIdx.x >> 5;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int r = q + 8 * it;
        tile[r][w] = (row0 + r < R && col0 + w < K) ? s[(row0 + r) * K + col0 + w] : (E)0;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int k = q + 8 * it;
        if (col0 + k < K && row0 + w < R) d[(col0 + k) * R + row0 + w] = tile[w][k];
    }
}

// One workgroup of an LDS-tiled kernel.  512 threads at most, so up to 256 VGPRs per lane.
template <class Kernel>
__global__ void __launch_bounds__(512) block_kernel_entry(typename Kernel::Params p)
{
    extern __shared__ __attribute__((aligned(16))) float ndc_lds[];
    DeviceExec<typename Kernel::State> ex;
    ex.lds = ndc_lds;
    ex.tid = threadIdx.x;
    ex.nthreads = blockDim.x;
    Kernel::run(ex, p, (int)blockIdx.x);
}

// The same for a kernel that declares `kWavesPerSimd = 4`: its LDS footprint lets four
// workgroups share a CU, so the register allocator is held to the 128 VGPRs that four
// wavefronts per SIMD leave each lane.
template <class Kernel>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
block_kernel_entry_w4(typename Kernel::Params p)
{
    extern __shared__ __attribute__((aligned(16))) float ndc_lds[];
    DeviceExec<typename Kernel::State> ex;
    ex.lds = ndc_lds;
    ex.tid = threadIdx.x;
    ex.nthreads = blockDim.x;
    Kernel::run(ex, p, (int)blockIdx.x);
}

template <class K, class = void> struct WavesWanted {
    static constexpr int value = 0;
};
template <class K> struct WavesWanted<K, decltype((void)K::kWavesPerSimd)> {
    static constexpr int value = K::kWavesPerSimd;
};

// Event stopwatch on one stream: mark() after each stage, finish() synchronises and
// reports the stage durations in milliseconds.
struct HipTimer {
    static const int kMax = 8;
    hipEvent_t ev[kMax + 1];
    int n = 0;
    bool on;
    hipStream_t stream;
    HipTimer(bool enable, void *s) : on(enable), stream((hipStream_t)s)
    {
        if (!on) return;
        for (int i = 0; i <= kMax; ++i) (void)hipEventCreate(&ev[i]);
        (void)hipEventRecord(ev[0], stream);
    }
    void mark()
    {
        if (on && n < kMax) (void)hipEventRecord(ev[++n], stream);
    }
    void finish(float *ms, int count)
    {
        if (!on) return;
        (void)hipEventSynchronize(ev[n]);
        for (int i = 0; i < count; ++i) {
            ms[i] = 0.f;
            if (i < n) (void)hipEventElapsedTime(&ms[i], ev[i], ev[i + 1]);
        }
        for (int i = 0; i <= kMax; ++i) (void)hipEventDestroy(ev[i]);
        on = false;
    }
    ~HipTimer() { if (on) for (int i = 0; i <= kMax; ++i) (void)hipEventDestroy(ev[i]); }
};

struct Backend {
    static constexpr bool is_device = true;
    typedef HipTimer Timer;

    template <class Kernel>
    static int block_kernel(const typename Kernel::Params &p, int nblocks, int nthreads,
                            int lds_floats, void *stream)
    {
        if (nblocks <= 0) return 0;
        const size_t bytes = (size_t)lds_floats * sizeof(float);
        void (*entry)(typename Kernel::Params) = block_kernel_entry<Kernel>;
        if constexpr (WavesWanted<Kernel>::value == 4) entry = block_kernel_entry_w4<Kernel>;
        if (bytes > 64 * 1024) {
            // more dynamic LDS than the default cap: raise it for this kernel (idempotent)
            if (hipFuncSetAttribute((const void *)entry, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)bytes) != hipSuccess)
                return -5;
        }
        hipLaunchKernelGGL(entry, dim3((unsigned)nblocks), dim3((unsigned)nthreads), bytes,
                           (hipStream_t)stream, p);
        return check();
    }

    static int check()
    {
        return hipGetLastError() == hipSuccess ? 0 : -5;
    }

    template <class F> static int elementwise(long long n, void *stream, F f)
    {
        if (n <= 0) return 0;
        long long blocks = (n + 255) / 256;
        if (blocks > (1LL << 20)) blocks = 1LL << 20;  // grid-stride beyond that
        hipLaunchKernelGGL(elementwise_kernel<F>, dim3((unsigned)blocks), dim3(256), 0,
                           (hipStream_t)stream, n, f);
        return check();
    }

    // dst[b][k][r] = src[b][r][k] for `batch` matrices of R x K elements of esz (2 or 4) bytes
    static int transpose(const void *src, void *dst, long long batch, long long R, long long K,
                         int esz, void *stream)
    {
        if (batch <= 0 || R <= 0 || K <= 0) return 0;
        const bool pairs = esz == 2 && R % 2 == 0 && K % 2 == 0 && (((uintptr_t)src | (uintptr_t)dst) & 3u) == 0;
        const long long t = pairs ? 64 : 32;
        const long long tiles_r = (R + t - 1) / t, tiles_k = (K + t - 1) / t;
        const long long nblk = batch * tiles_r * tiles_k;
        if (nblk > 0x7fffffffLL) return -2;
        if (pairs)
            hipLaunchKernelGGL(transpose_pairs_kernel, dim3((unsigned)nblk), dim3(256), 0, (hipStream_t)stream,
                               (const uint32_t *)src, (uint32_t *)dst, R, K, tiles_r, tiles_k);
        else if (esz == 2)
            hipLaunchKernelGGL(transpose_kernel<uint16_t>, dim3((unsigned)nblk), dim3(256), 0,
                               (hipStream_t)stream, (const uint16_t *)src, (uint16_t *)dst, R, K, tiles_r, tiles_k);
        else
            hipLaunchKernelGGL(transpose_kernel<uint32_t>, dim3((unsigned)nblk), dim3(256), 0,
                               (hipStream_t)stream, (const uint32_t *)src, (uint32_t *)dst, R, K, tiles_r, tiles_k);
        return check();
    }

    // ... one launch, a row per workgroup (held_kernel), where a row fits: the smallest workgroup that holds
    // it in a few vectors a thread.  Single elements (rows of no whole number of vectors): 8 or 16 a thread, so that
    // several small workgroups share a CU.  With 2 to 4 of them in 1024 threads a CU had some 8 KB in flight: us,
    // two launches -> 1024 threads -> as now, float32 forward: 8192 rows of 1025 28.7 -> 57.5 -> 15.6, of 2197 44.9 ->
    // 58.7 -> 24.1, of 4095 72.1 -> 63.3 -> 43.0; 256 rows of 2197 7.5 -> 4.7 -> 4.3.
    // False, with nothing launched, for rows that do not fit, and past the 2^32 threads of a launch.
    template <typename T, bool BWD, bool VEC, bool ADD, int PER, int NT>
    static bool rownorm_held_launch(const void *a, const void *b, const void *addend, float *stats, void *out, long long rows,
                                    long long n, float eps, void *stream)
    {
        if (rows > 0xffffffffLL / NT) return false;
        hipLaunchKernelGGL((rownorm::held_kernel<T, BWD, VEC, ADD, PER, NT>), dim3((unsigned)rows), dim3(NT), 0,
                           (hipStream_t)stream, (const T *)a, (const T *)b, (const T *)addend, (float2 *)stats, (T *)out, n, eps);
        return true;
    }
    template <typename T, bool BWD, bool VEC, bool ADD>
    static bool rownorm_held(const void *a, const void *b, const void *addend, float *stats, void *out, long long rows,
                             long long n, float eps, void *stream)
    {
        const long long nv = n / (VEC ? rownorm::Vec<T>::N : 1);
#define NDC_HELD(PER, NT) rownorm_held_launch<T, BWD, VEC, ADD, PER, NT>(a, b, addend, stats, out, rows, n, eps, stream)
        if (nv <= 2 * 64) return NDC_HELD(2, 64);
        if (nv <= 2 * 256) return NDC_HELD(2, 256);
        if (nv <= 4 * 256) return NDC_HELD(4, 256);
        // Long rows in vectors, few of them: one workgroup a row uses few CUs, and two launches read a row again from
        // the cache.  us, two launches -> held, forward and then forward + backward (the backward in two launches
        // either way: held it takes 8.6 against 8.1 on 64 rows of 32 768 floats): 64 rows of 24 000 floats 8.3 -> 6.3,
        // 17.2 -> 17.0; of 32 768 8.4 -> 7.2, 15.8 -> 17.6; 4 rows of 98 304 bf16 values 8.2 -> 8.5, 13.3 -> 14.1;
        // 96 rows of 65 536 10.3 -> 8.6, 22.0 -> 18.3.
        const bool few = VEC && rows < 96;
        const bool long_rows = nv <= (few ? 6 * 1024 : 8 * 1024) && (!BWD || rows >= 96);
        if constexpr (VEC) {
            if (nv <= 2 * 1024) return NDC_HELD(2, 1024);
            if (nv <= 4 * 1024) return NDC_HELD(4, 1024);
            if (long_rows) return NDC_HELD(8, 1024);
        } else {
            if (nv <= 8 * 256) return NDC_HELD(8, 256);
            if (nv <= 16 * 256) return NDC_HELD(16, 256);
            if (long_rows) return NDC_HELD(16, 512);
        }
        if constexpr (!BWD)
            if (nv <= 12 * 1024 && !few) return NDC_HELD(12, 1024);
#undef NDC_HELD
        return false;
    }

    // Row normalisation, one direction: reduce launch then apply launch on rows * nsplit
    // workgroups.  Forward: a = x, out = y, stats written; backward: a = gy, b = y, stats read,
    // out = gx.  `vec`: n is a multiple of 16 bytes of elements and every pointer is 16-byte
    // aligned.
    template <typename T, bool BWD, bool VEC>
    static void rownorm_launch(const void *a, const void *b, const void *addend, float *partial, float *stats,
                               void *out, long long rows, const rownorm::Split &sp, float eps, void *stream)
    {
        using namespace rownorm;
        if (BWD && addend ? rownorm_held<T, BWD, VEC, BWD>(a, b, addend, stats, out, rows, sp.n, eps, stream)
                          : rownorm_held<T, BWD, VEC, false>(a, b, nullptr, stats, out, rows, sp.n, eps, stream))
            return;
        const dim3 grid((unsigned)(rows * sp.nsplit)), block(kThreads);
        hipLaunchKernelGGL((reduce_kernel<T, BWD, VEC>), grid, block, 0, (hipStream_t)stream, (const T *)a,
                           (const T *)b, (float2 *)partial, sp);
        if (BWD && addend)
            hipLaunchKernelGGL((apply_kernel<T, BWD, VEC, BWD>), grid, block, 0, (hipStream_t)stream, (const T *)a,
                               (const T *)b, (const T *)addend, (const float2 *)partial, (float2 *)stats, (T *)out,
                               sp, eps);
        else
            hipLaunchKernelGGL((apply_kernel<T, BWD, VEC, false>), grid, block, 0, (hipStream_t)stream,
                               (const T *)a, (const T *)b, (const T *)nullptr, (const float2 *)partial,
                               (float2 *)stats, (T *)out, sp, eps);
    }

    // (mean, rstd) of every row
    static int rownorm_stats(const void *x, float *partial, float *stats, long long rows, long long n, int nsplit, long long chunk,
                             int esz, bool vec, float eps, void *stream)
    {
        using namespace rownorm;
        Split sp;
        sp.n = n, sp.nsplit = nsplit, sp.chunk = chunk;
        const dim3 grid((unsigned)(rows * nsplit)), block(kThreads);
        auto reduce = [&](auto kernel, auto *p) {
            hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, p, (decltype(p))nullptr, (float2 *)partial, sp);
        };
        if (esz == 2) vec ? reduce(reduce_kernel<bf16_t, false, true>, (const bf16_t *)x) : reduce(reduce_kernel<bf16_t, false, false>, (const bf16_t *)x);
        else vec ? reduce(reduce_kernel<float, false, true>, (const float *)x) : reduce(reduce_kernel<float, false, false>, (const float *)x);
        hipLaunchKernelGGL(stats_kernel, dim3((unsigned)((rows + kThreads - 1) / kThreads)), block, 0, (hipStream_t)stream,
                           (const float2 *)partial, (float2 *)stats, rows, sp, eps);
        return check();
    }

    // Row normalisation, one direction: reduce launch then apply launch on rows * nsplit
    // workgroups.  Forward: a = x, out = y, stats written; backward: a = gy, b = y, stats read,
    // out = gx (+ addend, if given).  `vec`: n is a multiple of 16 bytes of elements and every
    // pointer is 16-byte aligned.
    template <typename T>
    static void rownorm_t(bool bwd, const void *a, const void *b, const void *addend, float *partial, float *stats,
                          void *out, long long rows, const rownorm::Split &sp, bool vec, float eps, void *stream)
    {
        if (bwd) {
            if (vec) rownorm_launch<T, true, true>(a, b, addend, partial, stats, out, rows, sp, eps, stream);
            else rownorm_launch<T, true, false>(a, b, addend, partial, stats, out, rows, sp, eps, stream);
        } else {
            if (vec) rownorm_launch<T, false, true>(a, b, addend, partial, stats, out, rows, sp, eps, stream);
            else rownorm_launch<T, false, false>(a, b, addend, partial, stats, out, rows, sp, eps, stream);
        }
    }

    static int rownorm(bool bwd, const void *a, const void *b, const void *addend, float *partial, float *stats,
                       void *out, long long rows, long long n, int nsplit, long long chunk, int esz, bool vec,
                       float eps, void *stream)
    {
        if (rows <= 0 || n <= 0) return 0;
        const rownorm::Split sp = {n, chunk, nsplit};
        if (esz == 2) rownorm_t<bf16_t>(bwd, a, b, addend, partial, stats, out, rows, sp, vec, eps, stream);
        else rownorm_t<float>(bwd, a, b, addend, partial, stats, out, rows, sp, vec, eps, stream);
        return check();
    }

    // normalisation over the channels of a channel-first (B, C, n) tensor; see ndc_chnorm.h
    static constexpr int kChnormWaves = rownorm::kThreads / 64;   // partial rows per workgroup
    static long long chnorm_blocks(long long n, int esz, bool vec)
    {
        const long long per = vec ? 16 / esz : 1;
        return (n / per + rownorm::kThreads - 1) / rownorm::kThreads;
    }
    template <typename T, bool VEC>
    static void chnorm_launch(bool bwd, const void *a, const void *x, const float *stats, const float *weight,
                              const float *bias, void *out, float *partial, long long B, int C, long long n,
                              float eps, void *stream)
    {
        const chnorm::Shape sh = {n, C, (int)chnorm_blocks(n, (int)sizeof(T), VEC)};
        const dim3 grid((unsigned)(B * sh.blocks)), block(rownorm::kThreads);
        if (bwd)
            hipLaunchKernelGGL((chnorm::backward_kernel<T, VEC>), grid, block, 0, (hipStream_t)stream, (const T *)a,
                               (const T *)x, stats, weight, (T *)out, partial, sh);
        else
            hipLaunchKernelGGL((chnorm::forward_kernel<T, VEC>), grid, block, 0, (hipStream_t)stream, (const T *)x,
                               weight, bias, (T *)out, const_cast<float *>(stats), sh, eps);
    }
    // up to 256 channels: see held_forward_kernel.  Workgroups walk the voxels, 2048 of them in all
    // (two rounds of the chip at four a CU), never more than `partial` has rows.
    template <typename T, int LV, int CPT>
    static void chnorm_held_launch(bool bwd, const void *a, const void *x, const float *stats, const float *weight,
                                   const float *bias, void *out, float *partial, long long B, int C, long long n,
                                   long long parts, float eps, void *stream)
    {
        const long long tiles = (n / LV + 63) / 64, most = parts / B, want = (2048 + B - 1) / B;
        long long groups = tiles < want ? tiles : want;
        if (groups > most) groups = most;
        const chnorm::HeldShape sh = {n, C, (int)groups, tiles, parts};
        const dim3 grid((unsigned)(B * groups)), block(chnorm::kHeldThreads);
        if (bwd)
            hipLaunchKernelGGL((chnorm::held_backward_kernel<T, LV, CPT>), grid, block, 0, (hipStream_t)stream,
                               (const T *)a, (const T *)x, stats, weight, (T *)out, partial, sh);
        else
            hipLaunchKernelGGL((chnorm::held_forward_kernel<T, LV, CPT>), grid, block, 0, (hipStream_t)stream,
                               (const T *)x, weight, bias, (T *)out, const_cast<float *>(stats), sh, eps);
    }
    template <typename T, int LV>
    static void chnorm_held(bool bwd, const void *a, const void *x, const float *stats, const float *weight,
                            const float *bias, void *out, float *partial, long long B, int C, long long n,
                            long long parts, float eps, void *stream)
    {
        const int cpt = (C + chnorm::kSlices - 1) / chnorm::kSlices;
        if (cpt <= 4) chnorm_held_launch<T, LV, 4>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
        else if (cpt <= 8) chnorm_held_launch<T, LV, 8>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
        else if (cpt <= 16) chnorm_held_launch<T, LV, 16>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
        else chnorm_held_launch<T, LV, 32>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
    }

    // parts: rows of `partial` (ndc_chnorm_parts)
    static int chnorm(bool bwd, const void *a, const void *x, const float *stats, const float *weight,
                      const float *bias, void *out, float *partial, long long B, int C, long long n, int esz,
                      bool vec, long long parts, float eps, void *stream)
    {
        if (B <= 0 || C <= 0 || n <= 0) return 0;
        if (B * chnorm_blocks(n, esz, vec) > 0x7fffffffLL) return -2;
        if (C <= chnorm::kHeldChannels) {
            const bool pairs = n % 2 == 0 && (((uintptr_t)a | (uintptr_t)x | (uintptr_t)out) & (uintptr_t)(2 * esz - 1)) == 0;
            if (esz == 2 && pairs) chnorm_held<bf16_t, 2>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
            else if (esz == 2) chnorm_held<bf16_t, 1>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
            else if (pairs) chnorm_held<float, 2>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
            else chnorm_held<float, 1>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, parts, eps, stream);
            return check();
        }
        if (esz == 2) {
            if (vec) chnorm_launch<bf16_t, true>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, eps, stream);
            else chnorm_launch<bf16_t, false>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, eps, stream);
        } else {
            if (vec) chnorm_launch<float, true>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, eps, stream);
            else chnorm_launch<float, false>(bwd, a, x, stats, weight, bias, out, partial, B, C, n, eps, stream);
        }
        return check();
    }

    static int row_sums(const void *a, float *partial, long long rows, long long n, int nsplit, long long chunk,
                        int esz, bool vec, void *stream)
    {
        if (rows <= 0 || n <= 0) return 0;
        const rownorm::Split sp = {n, chunk, nsplit};
        const dim3 grid((unsigned)(rows * nsplit)), block(rownorm::kThreads);
        if (esz == 2) {
            if (vec) hipLaunchKernelGGL((rownorm::row_sums_kernel<bf16_t, true>), grid, block, 0, (hipStream_t)stream, (const bf16_t *)a, partial, sp);
            else hipLaunchKernelGGL((rownorm::row_sums_kernel<bf16_t, false>), grid, block, 0, (hipStream_t)stream, (const bf16_t *)a, partial, sp);
        } else {
            if (vec) hipLaunchKernelGGL((rownorm::row_sums_kernel<float, true>), grid, block, 0, (hipStream_t)stream, (const float *)a, partial, sp);
            else hipLaunchKernelGGL((rownorm::row_sums_kernel<float, false>), grid, block, 0, (hipStream_t)stream, (const float *)a, partial, sp);
        }
        return check();
    }

    // y = act(z + bias[channel]) + residual on rows * nsplit workgroups (bias, residual optional)
    template <typename T, int ACT, bool RES>
    static void bias_act_launch(const void *z, const float *bias, const void *res, void *y, int channels,
                                const rownorm::Split &sp, long long rows, bool vec, void *stream)
    {
        const dim3 grid((unsigned)(rows * sp.nsplit)), block(rownorm::kThreads);
        if (vec)
            hipLaunchKernelGGL((epilogue::forward_kernel<T, ACT, RES, true>), grid, block, 0, (hipStream_t)stream,
                               (const T *)z, bias, (const T *)res, (T *)y, channels, sp);
        else
            hipLaunchKernelGGL((epilogue::forward_kernel<T, ACT, RES, false>), grid, block, 0, (hipStream_t)stream,
                               (const T *)z, bias, (const T *)res, (T *)y, channels, sp);
    }

    template <typename T>
    static int bias_act_t(const void *z, const float *bias, const void *res, void *y, long long rows,
                          int channels, long long n, int nsplit, long long chunk, int act, bool vec, void *stream)
    {
        const rownorm::Split sp = {n, chunk, nsplit};
#define NDC_BIAS_ACT(ACT)                                                                        \
    (res ? bias_act_launch<T, ACT, true>(z, bias, res, y, channels, sp, rows, vec, stream)        \
         : bias_act_launch<T, ACT, false>(z, bias, res, y, channels, sp, rows, vec, stream))
        if (act == epilogue::kNone) NDC_BIAS_ACT(epilogue::kNone);
        else if (act == epilogue::kRelu) NDC_BIAS_ACT(epilogue::kRelu);
        else NDC_BIAS_ACT(epilogue::kGelu);
#undef NDC_BIAS_ACT
        return check();
    }

    static int bias_act(const void *z, const float *bias, const void *res, void *y, long long rows,
                        int channels, long long n, int nsplit, long long chunk, int act, int esz, bool vec,
                        void *stream)
    {
        if (rows <= 0 || n <= 0) return 0;
        return esz == 2 ? bias_act_t<bf16_t>(z, bias, res, y, rows, channels, n, nsplit, chunk, act, vec, stream)
                        : bias_act_t<float>(z, bias, res, y, rows, channels, n, nsplit, chunk, act, vec, stream);
    }

    template <typename T, int ACT>
    static void bias_act_bwd_launch(const void *gy, const void *z, const float *bias, void *gz, float *gpart,
                                    int channels, const rownorm::Split &sp, long long rows, bool vec, void *stream)
    {
        const dim3 grid((unsigned)(rows * sp.nsplit)), block(rownorm::kThreads);
        if (vec)
            hipLaunchKernelGGL((epilogue::backward_kernel<T, ACT, true>), grid, block, 0, (hipStream_t)stream,
                               (const T *)gy, (const T *)z, bias, (T *)gz, gpart, channels, sp);
        else
            hipLaunchKernelGGL((epilogue::backward_kernel<T, ACT, false>), grid, block, 0, (hipStream_t)stream,
                               (const T *)gy, (const T *)z, bias, (T *)gz, gpart, channels, sp);
    }

    // gz = gy * act'(z + bias), gpart[row * nsplit + part] = the part's sum of gz (act: relu, gelu)
    static int bias_act_backward(const void *gy, const void *z, const float *bias, void *gz, float *gpart,
                                 long long rows, int channels, long long n, int nsplit, long long chunk, int act,
                                 int esz, bool vec, void *stream)
    {
        if (rows <= 0 || n <= 0) return 0;
        const rownorm::Split sp = {n, chunk, nsplit};
        if (esz == 2) {
            if (act == epilogue::kRelu) bias_act_bwd_launch<bf16_t, epilogue::kRelu>(gy, z, bias, gz, gpart, channels, sp, rows, vec, stream);
            else bias_act_bwd_launch<bf16_t, epilogue::kGelu>(gy, z, bias, gz, gpart, channels, sp, rows, vec, stream);
        } else {
            if (act == epilogue::kRelu) bias_act_bwd_launch<float, epilogue::kRelu>(gy, z, bias, gz, gpart, channels, sp, rows, vec, stream);
            else bias_act_bwd_launch<float, epilogue::kGelu>(gy, z, bias, gz, gpart, channels, sp, rows, vec, stream);
        }
        return check();
    }

    // 2 x 2 (x 2) windows of a fine grid <-> 4 (8) planes of the coarse grid; see ndc_regroup.h
    static int regroup2(const void *src, void *dst, const float *bias, long long rows, int channels, int D,
                        int H, int W, int depth2, int esz, int to_channels, void *stream)
    {
        const regroup::Shape sh = {rows, D, H, W, depth2, channels};
        const long long nvec = rows * D * H * (W / (16 / esz));
        if (nvec <= 0) return 0;
        const long long blocks = (nvec + 255) / 256;
        if (blocks > 0x7fffffffLL) return -2;
        const dim3 grid((unsigned)blocks), block(256);
        if (esz == 2) {
            if (to_channels) hipLaunchKernelGGL((regroup::kernel<2, true>), grid, block, 0, (hipStream_t)stream, src, dst, bias, sh, nvec);
            else hipLaunchKernelGGL((regroup::kernel<2, false>), grid, block, 0, (hipStream_t)stream, src, dst, bias, sh, nvec);
        } else {
            if (to_channels) hipLaunchKernelGGL((regroup::kernel<4, true>), grid, block, 0, (hipStream_t)stream, src, dst, bias, sh, nvec);
            else hipLaunchKernelGGL((regroup::kernel<4, false>), grid, block, 0, (hipStream_t)stream, src, dst, bias, sh, nvec);
        }
        return check();
    }

    // weights (cout x cin, or the transpose stored as cin x cout) -> fragment order; see ndc_pwgemm.h
    static int pwgemm_pack(const void *w, int w_is_bf16, int transposed, void *wfrag, int cout, int cin, void *stream)
    {
        const long long n = (long long)(cout / 32) * (cin / 16) * 64;
        const dim3 grid((unsigned)((n + 255) / 256)), block(256);
        uint16_t *o = (uint16_t *)wfrag;
        if (w_is_bf16) {
            if (transposed) hipLaunchKernelGGL((pwgemm::pack_kernel<bf16_t, true>), grid, block, 0, (hipStream_t)stream, (const bf16_t *)w, o, cout, cin);
            else hipLaunchKernelGGL((pwgemm::pack_kernel<bf16_t, false>), grid, block, 0, (hipStream_t)stream, (const bf16_t *)w, o, cout, cin);
        } else {
            if (transposed) hipLaunchKernelGGL((pwgemm::pack_kernel<float, true>), grid, block, 0, (hipStream_t)stream, (const float *)w, o, cout, cin);
            else hipLaunchKernelGGL((pwgemm::pack_kernel<float, false>), grid, block, 0, (hipStream_t)stream, (const float *)w, o, cout, cin);
        }
        return check();
    }

    // persistent workgroups: as many as are resident at once (asked of the runtime once per
    // kernel and LDS size), so that every wavefront walks the same number of tiles
    template <int CIN, int ACT, bool RES, int THREADS, bool NORM = false>
    static int pwgemm_launch(const pwgemm::Params &p, size_t lds, void *stream)
    {
        void (*entry)(pwgemm::Params) = pwgemm::gemm_kernel<CIN, ACT, RES, THREADS, NORM>;
        static std::atomic<int> resident[3] = {{0}, {0}, {0}};   // by LDS size class
        const int cls = lds <= 40 * 1024 ? 0 : lds <= 80 * 1024 ? 1 : 2;
        int per_cu = resident[cls].load(std::memory_order_relaxed);
        if (per_cu == 0) {
            // (asked for the largest LDS size of the class, so that the answer holds for all of it)
            const size_t worst = cls == 0 ? 40 * 1024 : cls == 1 ? 80 * 1024 : 160 * 1024;
            if (worst > 64 * 1024 &&
                hipFuncSetAttribute((const void *)entry, hipFuncAttributeMaxDynamicSharedMemorySize, (int)worst) != hipSuccess)
                return -5;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)entry, THREADS, worst) != hipSuccess ||
                per_cu < 1)
                per_cu = 1;
            resident[cls].store(per_cu, std::memory_order_relaxed);
        }
        int dev = 0, cus = 256;
        if (hipGetDevice(&dev) == hipSuccess) {
            static std::atomic<int> cu_count{0};
            cus = cu_count.load(std::memory_order_relaxed);
            if (cus == 0) {
                if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
                cu_count.store(cus, std::memory_order_relaxed);
            }
        }
        long long blocks = (long long)cus * per_cu;
        const long long need = ((long long)p.tiles + THREADS / 64 - 1) / (THREADS / 64);
        if (blocks > need) blocks = need;
        // gradient modes: one row of sums per wavefront (the kernel zeroes the rows nobody owns)
        if (p.gpart && blocks * (THREADS / 64) > pwgemm::kMaxParts) blocks = pwgemm::kMaxParts / (THREADS / 64);
        hipLaunchKernelGGL(entry, dim3((unsigned)blocks), dim3(THREADS), lds, (hipStream_t)stream, p);
        return check();
    }

    template <int CIN, int THREADS>
    static int pwgemm_act(const pwgemm::Params &p, size_t lds, int act, void *stream)
    {
#define NDC_PWGEMM_RES(ACT)                                                                 \
    (p.res ? pwgemm_launch<CIN, ACT, true, THREADS>(p, lds, stream)                         \
           : pwgemm_launch<CIN, ACT, false, THREADS>(p, lds, stream))
        // gradient modes hold a row of sums per wavefront in LDS as well
        const size_t glds = lds + (size_t)(THREADS / 64) * p.cout * 4;
        if (act >= pwgemm::kReluGrad && glds > 160 * 1024) return -2;
        if (act == pwgemm::kGeluGrad) return pwgemm_launch<CIN, pwgemm::kGeluGrad, true, THREADS>(p, glds, stream);
        if (act == pwgemm::kReluGrad) return pwgemm_launch<CIN, pwgemm::kReluGrad, true, THREADS>(p, glds, stream);
        if (act == pwgemm::kMasked) return NDC_PWGEMM_RES(pwgemm::kMasked);
        if (act == epilogue::kRelu) return NDC_PWGEMM_RES(epilogue::kRelu);
        if (act == epilogue::kGelu) return NDC_PWGEMM_RES(epilogue::kGelu);
        return NDC_PWGEMM_RES(epilogue::kNone);
#undef NDC_PWGEMM_RES
    }

    // y = act(W x + bias) + residual on persistent workgroups; the caller has checked the shape
    // (cin in {32, 64, 128, 256}, cout a multiple of 32, n a multiple of 64, packed weights <= 128 KB)
    template <int CT, bool RES, bool MASK>
    static int pwgemm_deep_launch(const pwgemm::Params &p, int cin, size_t lds, void *stream)
    {
        constexpr int THREADS = 512;
        void (*entry)(pwgemm::Params, int) = pwgemm::gemm_kernel_deep<CT, RES, MASK, THREADS>;
        static std::atomic<int> resident[2] = {{0}, {0}};
        const int cls = lds <= 72 * 1024 ? 0 : 1;
        int per_cu = resident[cls].load(std::memory_order_relaxed);
        if (per_cu == 0) {
            const size_t worst = cls == 0 ? 72 * 1024 : 160 * 1024;
            if (hipFuncSetAttribute((const void *)entry, hipFuncAttributeMaxDynamicSharedMemorySize, (int)worst) != hipSuccess)
                return -5;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)entry, THREADS, worst) != hipSuccess ||
                per_cu < 1)
                per_cu = 1;
            resident[cls].store(per_cu, std::memory_order_relaxed);
        }
        int dev = 0, cus = 256;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
            cus = 256;
        long long blocks = (long long)cus * per_cu;
        const long long need = ((long long)p.tiles + THREADS / 64 - 1) / (THREADS / 64);
        if (blocks > need) blocks = need;
        hipLaunchKernelGGL(entry, dim3((unsigned)blocks), dim3(THREADS), lds, (hipStream_t)stream, p, cin);
        return check();
    }

    template <int CT>
    static int pwgemm_deep(const pwgemm::Params &p, int cin, size_t lds, void *stream)
    {
        if (p.mask)
            return p.res ? pwgemm_deep_launch<CT, true, true>(p, cin, lds, stream)
                         : pwgemm_deep_launch<CT, false, true>(p, cin, lds, stream);
        return p.res ? pwgemm_deep_launch<CT, true, false>(p, cin, lds, stream)
                     : pwgemm_deep_launch<CT, false, false>(p, cin, lds, stream);
    }

    // act 3 / 4: y = (W x) * relu' / gelu'(res + bias), gpart (kMaxParts x cout, or null) receives
    // per-wavefront sums of y whose total over the rows is the bias gradient
    // act 5: y = (W x + bias + res) where mask > 0, else 0
    static int pwgemm(const void *x, const void *wfrag, const float *bias, const void *res, void *y, void *zkeep,
                      float *gpart, const void *mask, long long batch, int cin, int cout, long long n, int act,
                      void *stream)
    {
        pwgemm::Params p = {};
        p.gpart = gpart;
        p.mask = (const uint16_t *)mask;
        p.x = (const uint16_t *)x, p.wfrag = (const uint16_t *)wfrag, p.bias = bias;
        p.res = (const uint16_t *)res, p.y = (uint16_t *)y, p.zkeep = (uint16_t *)zkeep;
        p.n = n, p.tiles_per_sample = (int)(n / pwgemm::kTileVoxels), p.tiles = (int)(batch * (n / pwgemm::kTileVoxels)), p.cout = cout;
        if (p.tiles <= 0) return 0;
        const size_t wbytes = (size_t)cin * cout * 2;
        const size_t lds = wbytes + (size_t)cout * 4;   // packed weights, bias
        if (cin > 256) {   // many input channels, at most 128 output channels (checked by the caller)
            if ((act != epilogue::kNone && act != pwgemm::kMasked) || zkeep) return -2;   // product, bias, residual, mask
            switch (cout / 32) {
            case 1: return pwgemm_deep<1>(p, cin, lds, stream);
            case 2: return pwgemm_deep<2>(p, cin, lds, stream);
            case 3: return pwgemm_deep<3>(p, cin, lds, stream);
            default: return pwgemm_deep<4>(p, cin, lds, stream);
            }
        }
        // small weight tables: several workgroups per CU; large ones: one, of more wavefronts
        int threads = wbytes <= 32 * 1024 ? 256 : wbytes <= 64 * 1024 || cin == 256 ? 512 : 1024;
        if (act >= pwgemm::kReluGrad && lds + (size_t)(threads / 64) * cout * 4 > 160 * 1024) threads = 512;
#define NDC_PWGEMM(CIN)                                                                            \
    (threads == 256 ? pwgemm_act<CIN, 256>(p, lds, act, stream)                                     \
     : threads == 512 ? pwgemm_act<CIN, 512>(p, lds, act, stream)                                   \
                      : pwgemm_act<CIN, 1024>(p, lds, act, stream))
        if (cin == 32) return NDC_PWGEMM(32);
        if (cin == 64) return NDC_PWGEMM(64);
        if (cin == 128) return NDC_PWGEMM(128);
        return threads == 256 ? pwgemm_act<256, 256>(p, lds, act, stream) : pwgemm_act<256, 512>(p, lds, act, stream);
#undef NDC_PWGEMM
    }

    // y = act(W normalised(x) + bias): the forms a block has (the caller has checked them)
    static int pwgemm_normed(const void *x, const float *stats, const void *wfrag, const float *bias, void *y, long long batch,
                             int cin, int cout, long long n, int act, void *stream)
    {
        pwgemm::Params p = {};
        p.x = (const uint16_t *)x, p.wfrag = (const uint16_t *)wfrag, p.bias = bias, p.y = (uint16_t *)y, p.stats = stats;
        p.n = n, p.tiles_per_sample = (int)(n / pwgemm::kTileVoxels), p.tiles = (int)(batch * (n / pwgemm::kTileVoxels)), p.cout = cout;
        const size_t lds = (size_t)cin * cout * 2 + (size_t)cout * 4;
        if (act == epilogue::kGelu) return pwgemm_launch<128, epilogue::kGelu, false, 1024, true>(p, lds, stream);
        if (cin == 32) return pwgemm_launch<32, epilogue::kRelu, false, 256, true>(p, lds, stream);
        if (cin == 64) return pwgemm_launch<64, epilogue::kRelu, false, 256, true>(p, lds, stream);
        return pwgemm_launch<128, epilogue::kRelu, false, 256, true>(p, lds, stream);
    }

    static int wgrad(const void *a, const void *b, float *gw, float *gb, float *part, long long batch, int rows, int cols,
                     long long n, int esz, const WgradPlan &plan, void *stream)
    {
        const int st = gemm::wgrad(a, b, gw, gb, part, batch, rows, cols, n, esz, plan, stream);
        return st ? st : check();
    }
    static int tile_gemm(const void *x, const float *w, int transposed, const float *bias, const void *res,
                         const void *mask, void *y, void *zkeep, float *gpart, long long batch, int cin, int cout,
                         long long n, int mode, int esz, int waves, void *stream)
    {
        const int st = gemm::tile_gemm(x, w, transposed, bias, res, mask, y, zkeep, gpart, batch, cin, cout, n, mode, esz, waves, stream);
        return st ? st : check();
    }

    static int mlp_forward(const void *x, const float *stats, const void *w1, const void *w2, int w_is_bf16, const float *b1,
                           const float *b2, const void *res, void *y, long long batch, int c, long long n, void *stream)
    {
        const int st = mlp::forward(x, stats, w1, w2, w_is_bf16, b1, b2, res, y, batch, c, n, stream);
        return st ? st : check();
    }
    static int mlp_backward(const void *x, const void *gy, const void *w1, const void *w2, int w_is_bf16, const float *b1,
                            void *gx, float *gw1, float *gb1, float *gw2, float *gb2, float *part, long long batch, int c,
                            long long n, void *stream)
    {
        const int st = mlp::backward(x, gy, w1, w2, w_is_bf16, b1, gx, gw1, gb1, gw2, gb2, part, batch, c, n, stream);
        return st ? st : check();
    }

    static int dice_bce_forward(const float *l, const float *y, float *loss, float *coef, float *partial, int rows, long long n,
                                int parts, long long chunk, void *stream)
    {
        hipLaunchKernelGGL(loss::sums_kernel, dim3((unsigned)(rows * parts)), dim3(loss::kThreads), 0, (hipStream_t)stream, l, y,
                           (float4 *)partial, n, parts, chunk);
        int log_width = 0;
        while ((1 << log_width) < parts && log_width < 6) ++log_width;
        hipLaunchKernelGGL(loss::finish_kernel, dim3(1), dim3(loss::kFinish), 0, (hipStream_t)stream, (const float4 *)partial,
                           (float2 *)coef, loss, rows, parts, log_width, 1.f / ((float)rows * (float)n));
        return check();
    }
    static int dice_bce_backward(const float *l, const float *y, const float *coef, const float *g, float *gl, int rows, long long n,
                                 int parts, long long chunk, void *stream)
    {
        hipLaunchKernelGGL(loss::grad_kernel, dim3((unsigned)(rows * parts)), dim3(loss::kThreads), 0, (hipStream_t)stream, l, y,
                           (const float2 *)coef, g, gl, n, parts, chunk, 1.f / ((float)rows * (float)n));
        return check();
    }

    static int adamw(const ndc_adamw_tensor *t, long long count, double lr, double beta1, double beta2, double eps, double decay,
                     void *stream)
    {
        adamw::Params q;
        q.beta1 = beta1, q.beta2 = beta2, q.lr = lr;
        q.decay = 1.0 - lr * decay, q.eps = (float)eps;
        q.count = 0;
        long long blocks = 0;
        auto flush = [&] {
            if (blocks) hipLaunchKernelGGL(adamw::update_kernel, dim3((unsigned)blocks), dim3(adamw::kThreads), 0, (hipStream_t)stream, q);
            q.count = 0, blocks = 0;
        };
        for (long long i = 0; i < count; ++i) {
            const long long need = (t[i].n + adamw::kChunk - 1) / adamw::kChunk;
            if (!need) continue;
            if (q.count == adamw::kTensors || blocks + need > 0x7fffffffLL) flush();
            q.t[q.count] = t[i], q.first[q.count] = (uint32_t)blocks;
            ++q.count, blocks += need;
        }
        flush();
        adamw::Steps s;
        for (long long i = 0; i < count; i += adamw::kSteps) {
            s.count = (int)(count - i < adamw::kSteps ? count - i : adamw::kSteps);
            for (int j = 0; j < s.count; ++j) s.step[j] = t[i + j].step;
            hipLaunchKernelGGL(adamw::count_kernel, dim3((unsigned)((s.count + 63) / 64)), dim3(64), 0, (hipStream_t)stream, s);
        }
        return check();
    }

    static constexpr int kSumSlices = 8;
    template <class P, class F> static int strided_sum(int nout, int nparts, void *stream, P put, F term)
    {
        if (nout <= 0) return 0;
        hipLaunchKernelGGL((strided_sum_kernel<P, F>), dim3((unsigned)((nout + 31) / 32)), dim3(256), 0,
                           (hipStream_t)stream, nout, nparts, put, term);
        return check();
    }

    template <class F> static int per_unit(long long units, long long npos, void *stream, F f)
    {
        const long long blocks = (npos + 127) / 128;
        if (units <= 0 || npos <= 0) return 0;
        if (blocks > 0x7fffffffLL / units) return -2;
        hipLaunchKernelGGL(per_unit_kernel<F>, dim3((unsigned)(units * blocks)), dim3(128), 0, (hipStream_t)stream,
                           (unsigned)blocks, npos, f);
        return check();
    }

    template <class F> static int weighted_unit(long long units, long long npos, void *stream, F f)
    {
        const long long blocks = (npos + 127) / 128;
        if (units <= 0 || npos <= 0) return 0;
        if (blocks > 0x7fffffffLL / units) return -2;
        const dim3 grid((unsigned)(units * blocks)), block(128);
        const int n = f.weights();
        if (F::Weights::staged(n, units * blocks * 2))
            hipLaunchKernelGGL((weighted_unit_kernel<F, true>), grid, block, (size_t)n * 4, (hipStream_t)stream, (unsigned)blocks, npos, f);
        else
            hipLaunchKernelGGL((weighted_unit_kernel<F, false>), grid, block, 0, (hipStream_t)stream, (unsigned)blocks, npos, f);
        return check();
    }

    template <class F> static int unit_sums(long long units, void *stream, F f)
    {
        if (units <= 0) return 0;
        if (units > 0x7fffffffLL) return -2;
        hipLaunchKernelGGL(unit_sums_kernel<F>, dim3((unsigned)units), dim3(256), 0, (hipStream_t)stream, f);
        return check();
    }
};

}  // namespace ndc

