// Launches of the tiled GEMMs; see ndc_gemm.h.
#include <hip/hip_runtime.h>

#include "ndc_gemm.h"
#include "ndc_gemm_host.h"

namespace ndc {
namespace gemm {

// the tile of a weight gradient's workgroup: rows x columns, by what the result holds
template <typename T, int WM, int WN, int RT, int CT, int D>
static void wgrad_launch(WgradParams p, void *stream)
{
    const unsigned blocks = 8u * (((unsigned)p.splits * (unsigned)(p.tiles_m * p.tiles_n) + 7u) / 8u);
    hipLaunchKernelGGL((wgrad_kernel<T, WM, WN, RT, CT, D>), dim3(blocks), dim3(64 * WM * WN), 0,
                       (hipStream_t)stream, p);
}
template <typename T, int D> static void wgrad_t(const WgradParams &p, int bm, int bn, void *stream)
{
    if (bm == 256) wgrad_launch<T, 4, 1, 2, 2, D>(p, stream);
    else if (bn == 256) wgrad_launch<T, 1, 4, 2, 2, D>(p, stream);
    else if (bm == 128 && bn == 128) wgrad_launch<T, 2, 2, 2, 2, D>(p, stream);
    else if (bm == 128) wgrad_launch<T, 4, 1, 1, 1, D>(p, stream);
    else if (bn == 128) wgrad_launch<T, 1, 4, 1, 1, D>(p, stream);
    else wgrad_launch<T, 2, 2, 1, 1, D>(p, stream);
}
int wgrad(const void *a, const void *b, float *gw, float *gb, float *part, long long batch, int rows, int cols,
                 long long n, int esz, const WgradPlan &plan, void *stream)
{
    WgradParams p;
    if (plan.per_sample == 0) {   // all voxels to a workgroup
        p.a = a, p.b = b, p.part = nullptr, p.gw = gw, p.gb = gb, p.n = n, p.rows = rows, p.cols = cols;
        p.tiles_m = (rows + plan.bm - 1) / plan.bm, p.tiles_n = (cols + plan.bn - 1) / plan.bn, p.splits = (int)batch;
        const dim3 grid((unsigned)(p.tiles_m * p.tiles_n)), block(64 * kWholeWaves);
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, p); };
        auto by_tile = [&](auto type, auto many) {
            typedef decltype(type) T;
            if (plan.bm == 32) launch(wgrad_whole_kernel<T, 32, decltype(many)::value>);
            else launch(wgrad_whole_kernel<T, 16, decltype(many)::value>);
        };
        auto by_samples = [&](auto type) {
            batch > (n * esz % 16 ? 3 : 8) ? by_tile(type, std::true_type()) : by_tile(type, std::false_type());
        };
        if (esz == 4) by_samples(0.f); else by_samples(bf16_t());
        return 0;
    }
    p.a = a, p.b = b, p.part = part, p.gw = gw, p.gb = gb, p.n = n, p.chunk = plan.chunk, p.rows = rows, p.cols = cols;
    p.tiles_m = (rows + plan.bm - 1) / plan.bm, p.tiles_n = (cols + plan.bn - 1) / plan.bn;
    p.per_sample = plan.per_sample, p.splits = (int)batch * plan.per_sample;
    if (esz == 4) wgrad_t<float, 8>(p, plan.bm, plan.bn, stream);
    else if (plan.depth == 16) wgrad_t<bf16_t, 16>(p, plan.bm, plan.bn, stream);
    else wgrad_t<bf16_t, 8>(p, plan.bm, plan.bn, stream);
    return 0;
}

template <typename T, bool WT, int MODE> static void tile_gemm_w(TileParams p, int waves, void *stream)
{
    if (waves <= 0) {   // small grid: channels sliced over the wavefronts, tiles of 32 or 16 rows
        const int rows = waves ? 16 : 32, step = 64 / rows * Gran<T>::E;
        int slices = (p.cin + step - 1) / step;
        if (slices > kMaxSlices) slices = kMaxSlices;
        p.tiles_m = (p.cout + rows - 1) / rows;
        p.tiles_n = (int)((p.n + 2 * rows - 1) / (2 * rows));
        const dim3 grid(8u * (unsigned)((p.tiles_m * p.tiles_n * p.batch + 7) / 8));
        if (waves) hipLaunchKernelGGL((sliced_kernel<T, WT, MODE, 16>), grid, dim3(64 * slices), 0, (hipStream_t)stream, p);
        else hipLaunchKernelGGL((sliced_kernel<T, WT, MODE, 32>), grid, dim3(64 * slices), 0, (hipStream_t)stream, p);
        return;
    }
    const int rows = 32 * waves;   // 32, 64 or 128 output rows per workgroup
    p.tiles_m = (p.cout + rows - 1) / rows;
    p.tiles_n = (int)((p.n + 127) / 128);
    // a launch takes fewer than 2^32 threads: as many samples at a time (2^20 of one voxel into 1024 channels are 2^32)
    auto launch = [&](auto kernel, unsigned threads) {
        const long long most = (0xffffffffLL / ((long long)threads * p.tiles_m) - 7) / p.tiles_n, batch = p.batch;
        TileParams q = p;
        for (long long b = 0; b < batch; b += q.batch) {
            q.batch = (int)(batch - b < most ? batch - b : most < 1 ? 1 : most);
            auto at = [&](auto *t, long long per) { return t ? (decltype(t))((char *)t + b * per * p.n * (long long)sizeof(T)) : t; };
            q.x = at(p.x, p.cin), q.res = at(p.res, p.cout), q.mask = at(p.mask, p.cout), q.y = at(p.y, p.cout);
            q.zkeep = at(p.zkeep, p.cout), q.gpart = p.gpart ? p.gpart + b * p.tiles_n * p.cout : nullptr;
            const dim3 grid(8u * (unsigned)(((long long)p.tiles_n * q.batch + 7) / 8) * (unsigned)p.tiles_m);
            hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, (hipStream_t)stream, q);
        }
    };
    if constexpr (sizeof(T) == 4) {
        // one chain of sums where it is no less exact than the float32 instruction was there (a grid that used to be
        // sliced had chains of eight channels)
        const long long sliced = (long long)p.batch * ((p.n + 63) / 64) * ((p.cout + 31) / 32);
        const bool one = p.cin <= 32 || (p.cin <= 64 && sliced > 1024);
        if (waves == 2) one ? launch(parts_kernel<WT, 2, false, MODE>, 256) : launch(parts_kernel<WT, 2, true, MODE>, 256);
        else one ? launch(parts_kernel<WT, 1, false, MODE>, 256) : launch(parts_kernel<WT, 1, true, MODE>, 256);
    } else {
        if (waves == 4) launch(tile_kernel<WT, 4, MODE>, 256);
        else if (waves == 2) launch(tile_kernel<WT, 2, MODE>, 128);
        else launch(tile_kernel<WT, 1, MODE>, 64);
    }
}
template <typename T>
static int tile_gemm_t(const TileParams &p, int transposed, int mode, int waves, void *stream)
{
    // (an activation follows a projection, whose weight lies as W; its derivative an input
    // gradient, whose weight lies as the transpose of what is applied)
    if (mode == epilogue::kNone && !transposed) tile_gemm_w<T, false, epilogue::kNone>(p, waves, stream);
    else if (mode == epilogue::kNone) tile_gemm_w<T, true, epilogue::kNone>(p, waves, stream);
    else if (mode == epilogue::kRelu && !transposed) tile_gemm_w<T, false, epilogue::kRelu>(p, waves, stream);
    else if (mode == epilogue::kGelu && !transposed) tile_gemm_w<T, false, epilogue::kGelu>(p, waves, stream);
    else if (mode == kGeluGrad && transposed) tile_gemm_w<T, true, kGeluGrad>(p, waves, stream);
    else return -2;
    return 0;
}
int tile_gemm(const void *x, const float *w, int transposed, const float *bias, const void *res,
                     const void *mask, void *y, void *zkeep, float *gpart, long long batch, int cin, int cout, long long n,
                     int mode, int esz, int waves, void *stream)
{
    TileParams p;
    p.gpart = gpart, p.x = x, p.w = w, p.bias = bias, p.res = res, p.mask = mask, p.y = y, p.zkeep = zkeep, p.n = n, p.cin = cin;
    p.cout = cout, p.batch = (int)batch;
    return esz == 2 ? tile_gemm_t<bf16_t>(p, transposed, mode, waves, stream)
                    : tile_gemm_t<float>(p, transposed, mode, waves, stream);
}

}  // namespace gemm
}  // namespace ndc
