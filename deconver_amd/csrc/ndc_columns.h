// The column matrix of a convolution with few input channels (ndc_columns): every tap's shifted copy
// of the zero-padded grid, V voxels of one row per thread, stored with one access.  It writes taps
// times what it reads, so stores bound it; the shifted loads come out of the caches.  One launch:
// padding, a strided copy per tap and their concatenation before (2 channels of 96 x 128 x 112 in
// bfloat16: 28 launches, 0.20 ms; 0.073 here for the 149 MB it writes, of which the loads of a
// thread's eight voxels one by one are the larger part).
#pragma once
#include "ndc_direct.h"

namespace ndc {

template <typename E, int V> struct Columns {
    KGeom q;             // (D, H, W), the kernel and its padding
    const E *src;
    E *dst;
    struct alignas(V * sizeof(E)) Group {
        E v[V];
    };
    // unit: (row, tap); position: a group of V voxels
    NDC_HD void operator()(int u, long long pos) const
    {
        const int tap = u % q.KT, row = u / q.KT;
        const int tw = tap % q.kW, th = tap / q.kW % q.kH, td = tap / q.kW / q.kH;
        const direct::Pos<uint32_t> p = direct::position<uint32_t>(q, (uint32_t)pos * V);
        const int d = p.d + td - q.pD, h = p.h + th - q.pH, w = p.w + tw - q.pW;
        const bool in = (unsigned)d < (unsigned)q.D && (unsigned)h < (unsigned)q.H;
        const E *line = src + row * q.SP + (in ? ((long long)d * q.H + h) * q.W : 0);
        Group g;
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const bool here = in && (unsigned)(w + j) < (unsigned)q.W;
            const E v = line[here ? w + j : 0];
            g.v[j] = here ? v : (E)0;
        }
        *reinterpret_cast<Group *>(dst + (long long)u * q.SP + pos * V) = g;
    }
};

}  // namespace ndc
