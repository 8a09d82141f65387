// Launches of the MLP kernels (ndc_mlp.hip), kept apart from the kernels so that the library's
// translation units compile side by side.
#pragma once
#include <stddef.h>

namespace ndc {
namespace mlp {

static const int kTileVoxels = 64;   // voxels a wavefront (forward) or workgroup (backward) takes at a time
static const int kGradGroups = 256;  // workgroups of the backward: one per CU

// float32 partial results of one workgroup of the backward: gw1, gw2, gb1, four rows of gb2
static constexpr long long part_floats(int c) { return 8LL * c * c + 4LL * c + 4LL * c; }
static inline int grad_groups(long long tiles) { return tiles < kGradGroups ? (int)tiles : kGradGroups; }

// w1 (4 c, c), w2 (c, 4 c) as they lie, float32 or bf16; res may be null, with stats (the rows' (mean, 1 /
// deviation), x is normalised by them) it may not; the caller checks the launch
int forward(const void *x, const float *stats, const void *w1, const void *w2, int w_is_bf16, const float *b1, const float *b2,
            const void *res, void *y, long long batch, int c, long long n, void *stream);
int backward(const void *x, const void *gy, const void *w1, const void *w2, int w_is_bf16, const float *b1, void *gx,
             float *gw1, float *gb1, float *gw2, float *gb2, float *part, long long batch, int c, long long n, void *stream);

}  // namespace mlp
}  // namespace ndc
