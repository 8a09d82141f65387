// Launches of the tiled GEMMs (ndc_gemm.hip), kept apart from their kernels so that the library's
// translation units compile side by side.
#pragma once

namespace ndc {

// how ndc_weight_grad cuts its work: tile of the result per workgroup, stage depth in granules,
// voxels per split
struct WgradPlan {
    int bm, bn, depth, per_sample;   // per_sample 0: all samples and voxels in one workgroup
    long long chunk;
};

namespace gemm {

// 0, or -2 for a combination that has no kernel; the caller checks the launch
int wgrad(const void *a, const void *b, float *gw, float *gb, float *part, long long batch, int rows, int cols, long long n,
          int esz, const WgradPlan &plan, void *stream);
int tile_gemm(const void *x, const float *w, int transposed, const float *bias, const void *res, const void *mask, void *y,
              void *zkeep, float *gpart, long long batch, int cin, int cout, long long n, int mode, int esz, int waves,
              void *stream);

}  // namespace gemm
}  // namespace ndc
