// Launches of the MLP kernels; see ndc_mlp.h.
#include <hip/hip_runtime.h>

#include "ndc_mlp.h"

namespace ndc {
namespace mlp {

static Params params(const void *x, const void *w1, const void *w2, const float *b1, void *y, long long batch, long long n)
{
    Params p = {};
    p.x = (const uint16_t *)x, p.w1 = w1, p.w2 = w2, p.b1 = b1, p.y = (uint16_t *)y, p.n = n;
    p.tiles_per_sample = (int)(n / kTileVoxels), p.tiles = (int)(batch * (n / kTileVoxels));
    return p;
}

template <int C, typename TW, int THREADS, bool HALF = false> static void forward_launch_t(const Params &p, int per_cu, void *stream)
{
    const int at_once = THREADS / 64 / (HALF ? 2 : 1), need = (p.tiles + at_once - 1) / at_once;
    const int blocks = need < 256 * per_cu ? need : 256 * per_cu;
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(THREADS), 0, (hipStream_t)stream, p); };
    if (p.stats) launch(forward_kernel<C, TW, true, THREADS, true, HALF>);
    else if (p.res) launch(forward_kernel<C, TW, true, THREADS, false, HALF>);
    else launch(forward_kernel<C, TW, false, THREADS, false, HALF>);
}
// A tile keeps its SIMD's vector unit busy for about 10 us at C = 64 (a third of that at 32), so few tiles go
// to workgroups small enough to reach all CUs: with twelve wavefronts each, 512 tiles ran 36 us on 43 CUs.
// At C = 32, up to one tile for two SIMDs, a tile goes to two wavefronts: 4096 voxels 10.0 -> 7.5 us (the two
// projections 8.1), 32 768 10.4 -> 8.2.
template <int C, typename TW> static void forward_launch(const Params &p, void *stream)
{
    if constexpr (C == 32) {
        if (p.tiles <= 512) forward_launch_t<C, TW, 256, true>(p, 4, stream);
        else forward_launch_t<C, TW, 256>(p, 4, stream);
    }
    else if (p.tiles <= 4 * 256) forward_launch_t<C, TW, 256>(p, 2, stream);
    else if (p.tiles <= 8 * 256) forward_launch_t<C, TW, 512>(p, 1, stream);
    else forward_launch_t<C, TW, 768>(p, 1, stream);
}

int forward(const void *x, const float *stats, const void *w1, const void *w2, int w_is_bf16, const float *b1, const float *b2,
            const void *res, void *y, long long batch, int c, long long n, void *stream)
{
    Params p = params(x, w1, w2, b1, y, batch, n);
    p.b2 = b2, p.res = (const uint16_t *)res, p.stats = stats;
    if (c == 64) {
        if (w_is_bf16) forward_launch<64, bf16_t>(p, stream);
        else forward_launch<64, float>(p, stream);
    } else if (c == 32) {
        if (w_is_bf16) forward_launch<32, bf16_t>(p, stream);
        else forward_launch<32, float>(p, stream);
    } else {
        return -2;
    }
    return 0;
}

template <int C, typename TW>
static void backward_launch(const Params &p, float *gw1, float *gb1, float *gw2, float *gb2, void *stream)
{
    const int groups = grad_groups(p.tiles), values = 8 * C * C + 4 * C + C;
    const bool g1 = gw1 || gb1, g2 = gw2 || gb2;
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(groups), dim3(8 * C), 0, (hipStream_t)stream, p); };
    // (some of the gradients: us, forward + backward with all -> these, 64 channels over 32 768 voxels: x's alone
    // 61.7 -> 32.8, the second projection's 61.0 -> 50.1)
    if (!g1 && !g2) launch(backward_kernel<C, TW, true, false, false>);
    else if (!p.y && !g1) launch(backward_kernel<C, TW, false, false, true>);
    else launch(backward_kernel<C, TW, true, true, true>);
    if (g1 || g2)
        hipLaunchKernelGGL((sum_kernel<C>), dim3((values + 127) / 128), dim3(256), 0, (hipStream_t)stream, p.part, groups, gw1, gb1, gw2,
                           gb2);
}

int backward(const void *x, const void *gy, const void *w1, const void *w2, int w_is_bf16, const float *b1, void *gx,
             float *gw1, float *gb1, float *gw2, float *gb2, float *part, long long batch, int c, long long n, void *stream)
{
    Params p = params(x, w1, w2, b1, gx, batch, n);
    p.gy = (const uint16_t *)gy, p.part = part;
    if (c == 64) {
        if (w_is_bf16) backward_launch<64, bf16_t>(p, gw1, gb1, gw2, gb2, stream);
        else backward_launch<64, float>(p, gw1, gb1, gw2, gb2, stream);
    } else if (c == 32) {
        if (w_is_bf16) backward_launch<32, bf16_t>(p, gw1, gb1, gw2, gb2, stream);
        else backward_launch<32, float>(p, gw1, gb1, gw2, gb2, stream);
    } else {
        return -2;
    }
    return 0;
}

}  // namespace mlp
}  // namespace ndc
