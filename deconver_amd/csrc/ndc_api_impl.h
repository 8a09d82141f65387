// Host-side logic of the C ABI (include/deconver_ndc.h): argument checks, path choice,
// workspace carving, launch sequence.  Included by exactly two translation units, each of
// which first defines a `Backend` with the launch primitives:
//   ndc_capi.hip       -> HIP launches on gfx950 (the product)
//   ndc_hostcheck.cpp  -> sequential host execution of the same kernel bodies (CPU tests)
#pragma once

#include "../../include/deconver_ndc.h"
#include "ndc_common.h"
#include "ndc_columns.h"
#include "ndc_direct_tile.h"
#include "ndc_fused_api.h"
#include "ndc_mlp_host.h"

namespace ndc {

static inline int make_kgeom(const ndc_geom *g, KGeom &q)
{
    if (!g) return NDC_ERR_NULL;
    if (g->dtype != NDC_F32 && g->dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (g->batch < 1 || g->groups < 1 || g->m < 1 || g->sc < 1) return NDC_ERR_GEOMETRY;
    long long taps = 1, sp = 1;
    for (int a = 0; a < 3; ++a) {
        if (g->size[a] < 1 || g->kernel[a] < 1 || (g->kernel[a] & 1) == 0) return NDC_ERR_GEOMETRY;
        taps *= g->kernel[a];
        sp *= g->size[a];
    }
    if (taps > 4096 || g->m > 1024 || g->sc > 1024) return NDC_ERR_GEOMETRY;
    // element counts must stay well inside int64 and block counts inside int32
    const long long cmax = (long long)g->groups * (g->m > g->sc ? g->m : g->sc);
    if (sp > (1LL << 40) || (long double)sp * cmax * g->batch > 9.0e15L) return NDC_ERR_GEOMETRY;
    if (g->path < NDC_PATH_AUTO || g->path > NDC_PATH_FUSED_VECTOR) return NDC_ERR_GEOMETRY;
    q.B = g->batch;
    q.G = g->groups;
    q.m = g->m;
    q.sc = g->sc;
    q.D = g->size[0];
    q.H = g->size[1];
    q.W = g->size[2];
    q.kD = g->kernel[0];
    q.kH = g->kernel[1];
    q.kW = g->kernel[2];
    q.pD = q.kD / 2;
    q.pH = q.kH / 2;
    q.pW = q.kW / 2;
    q.KT = (int)taps;
    q.relu = g->relu_input ? 1 : 0;
    // the kernel family is fixed here, once per call: named by the call, or the process default
    q.matrix = g->path == NDC_PATH_FUSED_MATRIX   ? 1
               : g->path == NDC_PATH_FUSED_VECTOR ? 0
                                                  : fused::matrix_default().load(std::memory_order_relaxed);
    q.gate = 0;
    q.eps = g->eps;
    q.SP = sp;
    return NDC_OK;
}

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Decide which implementation serves a call.  Returns NDC_PATH_DIRECT / NDC_PATH_FUSED, or
// a negative status when the caller forced a path that does not cover the geometry.
static inline int choose_path(const ndc_geom *g, const KGeom &q)
{
    const bool fused_ok = fused::supported(q);
    if (g->path == NDC_PATH_DIRECT) return NDC_PATH_DIRECT;
    if (g->path == NDC_PATH_FUSED || g->path == NDC_PATH_FUSED_MATRIX || g->path == NDC_PATH_FUSED_VECTOR)
        return fused_ok ? (int)NDC_PATH_FUSED : (int)NDC_ERR_GEOMETRY;
    return fused_ok ? (int)NDC_PATH_FUSED : (int)NDC_PATH_DIRECT;
}

// ------------------------------------------------------------------ direct path

template <typename TI, typename TO>
static int direct_gconv(const KGeom &q, const TI *in, const float *h, const float *bias,
                        int adjoint, TO *out, void *stream)
{
    const int rectify = bias != nullptr || q.relu, cout = adjoint ? q.sc : q.m;
    return direct::with_form(q, cout, [&](auto form) {
        typedef decltype(form) F;
        const int blocks = (cout + F::nb - 1) / F::nb;
        const long long units = (long long)q.B * q.G * blocks;
        if (adjoint) {
            const direct::GConv<TI, TO, true, F::nb, F::kwb, typename F::off> op = {q, in, h, bias, rectify, out, blocks};
            return direct::launch<Backend>(op, units, stream);
        }
        const direct::GConv<TI, TO, false, F::nb, F::kwb, typename F::off> op = {q, in, h, bias, rectify, out, blocks};
        return direct::launch<Backend>(op, units, stream);
    });
}

// n = A(x) + eps, d = A(t1) + eps and what STAGE makes of them (ndc_direct.h)
template <typename T, int STAGE>
static int direct_ratio(const KGeom &q, const T *x, const T *t1, const T *z, const T *gout, const float *gt1,
                        const float *h, const float *bias, T *out, T *s_over_den, T *ratio, float *gn, float *gd,
                        void *stream)
{
    return direct::with_form(q, q.sc, [&](auto form) {
        typedef decltype(form) F;
        const int blocks = (q.sc + F::nb - 1) / F::nb;
        const direct::Ratio<T, STAGE, F::nb, F::kwb, typename F::off> op = {
            q, x, t1, z, gout, gt1, h, bias, out, s_over_den, ratio, gn, gd, blocks};
        return direct::launch<Backend>(op, (long long)q.B * q.G * blocks, stream);
    });
}

template <typename T>
static int direct_forward(const KGeom &q, const T *x, const T *z, const float *h,
                          const float *bias, T *out, T *t1, T *s_over_den, T *ratio, void *stream)
{
    // t1 = K(relu(z + b)) lands in the caller's t1; without one there is nowhere to put
    // it, so the direct path asks for it (the fused path does not need it)
    if (!t1) return NDC_ERR_NULL;
    int st = direct_gconv<T, T>(q, z, h, bias, 0, t1, stream);
    if (st) return st;
    return direct_ratio<T, direct::FWD>(q, x, t1, z, nullptr, nullptr, h, bias, out, s_over_den, ratio, nullptr,
                                        nullptr, stream);
}

static inline size_t direct_backward_ws(const KGeom &q)
{
    const size_t n_x = (size_t)q.B * q.C() * q.SP, n_s = (size_t)q.B * q.CS() * q.SP;
    const size_t sums = (size_t)q.G * q.m * q.sc * q.KT + q.CS();
    return align_up(n_s * 4, 256) * 2 + align_up(n_x * 4, 256) +
           align_up((size_t)direct::reduce_chunks(q) * sums * 4, 256);
}

// scratch: gn | gd | gt1 (all float) | partial sums of gh and gb, [chunk][gh, gb]
template <typename T>
static int direct_backward(const KGeom &q, const T *x, const T *z, const T *t1, const float *h,
                           const float *bias, const T *gout, T *gx, T *gz, float *gh, float *gb,
                           void *ws, void *stream)
{
    const long long n_x = (long long)q.B * q.C() * q.SP, n_s = (long long)q.B * q.CS() * q.SP;
    char *w = (char *)ws;
    float *gn = (float *)w;
    w += align_up((size_t)n_s * 4, 256);
    float *gd = (float *)w;
    w += align_up((size_t)n_s * 4, 256);
    float *gt1 = (float *)w;
    w += align_up((size_t)n_x * 4, 256);
    float *part = (float *)w;
    const int n_gh = q.G * q.m * q.sc * q.KT, nchunk = direct::reduce_chunks(q);
    const long long stride = (long long)n_gh + q.CS();
    KGeom qn = q;  // gn/gd/gt1 are plain tensors: no bias, no rectification on load
    qn.relu = 0;
    int st = direct_ratio<T, direct::GRAD>(q, x, t1, z, gout, nullptr, h, bias, nullptr, nullptr, nullptr, gn, gd,
                                           stream);
    if (st) return st;
    if (!gx) {
        st = direct_gconv<float, float>(qn, gd, h, nullptr, 0, gt1, stream);
    } else {
        st = direct::with_form(q, q.m, [&](auto form) {
            typedef decltype(form) F;
            const int blocks = (q.m + F::nb - 1) / F::nb;
            const direct::GradPair<T, F::nb, F::kwb, typename F::off> op = {q, gn, gd, h, gx, gt1, blocks};
            return direct::launch<Backend>(op, (long long)q.B * q.G * blocks, stream);
        });
    }
    if (st) return st;
    if (gh) {
        st = direct::with_grad_form(q, [&](auto form) {
            typedef decltype(form) F;
            const int ob = (q.m + F::mb - 1) / F::mb, ib = (q.sc + F::sb - 1) / F::sb, wb = q.kW / F::kwb;
            const direct::FilterGrad<T, F::mb, F::sb, F::kwb, typename F::off> op = {
                q, x, t1, z, bias, gn, gd, gt1, part, stride, nchunk, ob, ib, wb};
            return Backend::unit_sums((long long)q.G * ob * ib * q.kD * q.kH * wb * nchunk, stream, op);
        });
        if (st) return st;
    }
    if (gz || gb) {
        // gz is needed to form gb; when the caller does not want gz it goes to the gn
        // scratch (gn is dead by now), typed as T
        T *gz_out = gz ? gz : (T *)gn;
        st = direct_ratio<T, direct::SOURCE>(q, x, t1, z, gout, gt1, h, bias, gz_out, nullptr, nullptr, nullptr,
                                             nullptr, stream);
        if (st) return st;
        if (gb) {
            const direct::BiasGrad<T> op = {q, gz_out, part + n_gh, stride, nchunk};
            st = Backend::unit_sums((long long)q.CS() * nchunk, stream, op);
            if (st) return st;
        }
    }
    // the chunks' sums, added in order (no atomics: results are reproducible)
    const int lo = gh ? 0 : n_gh, n = (gh ? n_gh : 0) + (gb ? q.CS() : 0), gate = q.gate;
    if (!n) return NDC_OK;
    return Backend::strided_sum(n, nchunk, stream, [=] NDC_LAMBDA(int o, float v) {
        if (lo + o < n_gh) gh[o] = gate && h[o] <= 0.f ? 0.f : v; else gb[lo + o - n_gh] = v;
    }, [=] NDC_LAMBDA(int o, int p) { return part[p * stride + lo + o]; });
}

}  // namespace ndc

// ============================================================================ C ABI

extern "C" {

int ndc_version(void) { return 300; }   // 0.3.0: the projections themselves (streaming GEMM)

const char *ndc_status_string(int status)
{
    switch (status) {
    case NDC_OK: return "ok";
    case NDC_ERR_NULL: return "a required pointer is null";
    case NDC_ERR_GEOMETRY: return "geometry not covered by the requested path";
    case NDC_ERR_DTYPE: return "unknown dtype tag";
    case NDC_ERR_WORKSPACE: return "workspace too small or misaligned";
    case NDC_ERR_LAUNCH: return "kernel launch failed";
    case NDC_ERR_SCRATCH_LIMIT:
        return "geometry needs more scratch than the no-allocation entry point's device array holds";
    default: return "unknown status";
    }
}

int ndc_fused_supported(const ndc_geom *g)
{
    ndc::KGeom q;
    if (ndc::make_kgeom(g, q) != NDC_OK) return 0;
    return ndc::fused::supported(q) ? 1 : 0;
}

int ndc_check_geometry(const ndc_geom *g)
{
    ndc::KGeom q;
    int st = ndc::make_kgeom(g, q);
    if (st) return st;
    st = ndc::choose_path(g, q);
    return st < 0 ? st : NDC_OK;
}

size_t ndc_forward_workspace_bytes(const ndc_geom *g)
{
    using namespace ndc;
    KGeom q;
    if (make_kgeom(g, q) != NDC_OK) return 0;
    const int path = choose_path(g, q);
    if (path != NDC_PATH_FUSED) return 0;
    return fused::forward_ws(q, g->dtype);
}

size_t ndc_taps_bytes(const ndc_geom *g) { return ndc_forward_workspace_bytes(g); }

int ndc_prepare_taps(const ndc_geom *g, const float *h, void *taps, size_t taps_bytes, void *stream)
{
    using namespace ndc;
    KGeom q;
    const int st = make_kgeom(g, q);
    if (st) return st;
    const size_t need = ndc_taps_bytes(g);
    if (!need) return NDC_OK;
    if (!h) return NDC_ERR_NULL;
    if (!taps || taps_bytes < need || ((uintptr_t)taps & 255u)) return NDC_ERR_WORKSPACE;
    return fused::prepare_taps<Backend>(q, h, (float *)taps, stream);
}

// What the layer's node had as passes of its own, some 3 to 4 us on the GPU and 5 to 8 of the host's each: the filter's
// rectifier rides on the launch that packs the table (one of the library's own where there is none), its backward on
// the launch that adds up gh.  3-D training step on one 32^3 volume 3.85 -> 3.75 ms, a block of 64 channels of
// 44 x 52 x 60 851 -> 847 us, a grouped layer of 24^3 206.6 -> 205.8.
int ndc_rectify_filter(const ndc_geom *g, const float *h0, float *h, void *taps, size_t taps_bytes, void *stream)
{
    using namespace ndc;
    KGeom q;
    const int st = make_kgeom(g, q);
    if (st) return st;
    if (!h0 || !h) return NDC_ERR_NULL;
    const size_t need = ndc_taps_bytes(g);
    if (!need || !taps)
        return Backend::elementwise((long long)q.G * q.m * q.sc * q.KT, stream,
                                    [=] NDC_LAMBDA(long long i) { h[i] = floor_f(h0[i], 0.f); });
    if (taps_bytes < need || ((uintptr_t)taps & 255u)) return NDC_ERR_WORKSPACE;
    return fused::rectify_and_prepare<Backend>(q, h0, h, (float *)taps, stream);
}

static int forward_impl(const ndc_geom *g, const void *x, const void *z, const float *h,
                        const float *bias, void *out, void *t1, void *s_over_den, void *ratio,
                        const void *taps, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace ndc;
    KGeom q;
    int st = make_kgeom(g, q);
    if (st) return st;
    if (!x || !z || !h || !out) return NDC_ERR_NULL;
    if ((s_over_den == nullptr) != (ratio == nullptr)) return NDC_ERR_NULL;
    const int path = choose_path(g, q);
    if (path < 0) return path;
    if (path == NDC_PATH_FUSED) {
        const size_t need = taps ? 0 : fused::forward_ws(q, g->dtype);
        if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255u)))
            return NDC_ERR_WORKSPACE;
        void *ws = need ? workspace : nullptr;
        const float *tp = fused::forward_ws(q, g->dtype) ? (const float *)taps : nullptr;
        return g->dtype == NDC_F32
                   ? fused::forward<Backend, float>(q, (const float *)x, (const float *)z, h, bias,
                                                    (float *)out, (float *)t1, (float *)s_over_den,
                                                    (float *)ratio, tp, ws, stream)
                   : fused::forward<Backend, bf16_t>(q, (const bf16_t *)x, (const bf16_t *)z, h,
                                                     bias, (bf16_t *)out, (bf16_t *)t1,
                                                     (bf16_t *)s_over_den, (bf16_t *)ratio, tp, ws,
                                                     stream);
    }
    return g->dtype == NDC_F32
               ? direct_forward<float>(q, (const float *)x, (const float *)z, h, bias,
                                       (float *)out, (float *)t1, (float *)s_over_den,
                                       (float *)ratio, stream)
               : direct_forward<bf16_t>(q, (const bf16_t *)x, (const bf16_t *)z, h, bias,
                                        (bf16_t *)out, (bf16_t *)t1, (bf16_t *)s_over_den,
                                        (bf16_t *)ratio, stream);
}

int ndc_forward(const ndc_geom *g, const void *x, const void *z, const float *h,
                const float *bias, void *out, void *t1, void *s_over_den, void *ratio,
                void *workspace, size_t workspace_bytes, void *stream)
{
    return forward_impl(g, x, z, h, bias, out, t1, s_over_den, ratio, nullptr, workspace,
                        workspace_bytes, stream);
}

int ndc_forward_taps(const ndc_geom *g, const void *x, const void *z, const float *h,
                     const void *taps, const float *bias, void *out, void *t1, void *s_over_den,
                     void *ratio, void *stream)
{
    if (ndc_taps_bytes(g) && (!taps || ((uintptr_t)taps & 255u))) return NDC_ERR_WORKSPACE;
    return forward_impl(g, x, z, h, bias, out, t1, s_over_den, ratio, taps, nullptr, 0, stream);
}

int ndc_matrix_kernels(int on)
{
    if (on >= 0) ndc::fused::matrix_default().store(on ? 1 : 0, std::memory_order_relaxed);
    return ndc::fused::matrix_default().load(std::memory_order_relaxed);
}

int ndc_backward_uses_saved(const ndc_geom *g)
{
    using namespace ndc;
    KGeom q;
    if (!g || make_kgeom(g, q) != NDC_OK) return 0;
    if (choose_path(g, q) != NDC_PATH_FUSED) return 0;
    return fused::backward_uses_saved(q, g->dtype) ? 1 : 0;
}

size_t ndc_backward_workspace_bytes(const ndc_geom *g, int need_gx, int need_gz, int need_gh,
                                    int need_gb)
{
    using namespace ndc;
    KGeom q;
    if (make_kgeom(g, q) != NDC_OK) return 0;
    const int path = choose_path(g, q);
    if (path < 0) return 0;
    (void)need_gx;
    (void)need_gz;
    if (path == NDC_PATH_FUSED) return fused::backward_ws(q, g->dtype, need_gh, need_gb);
    return direct_backward_ws(q);
}

static int backward_impl(const ndc_geom *g, const void *x, const void *z, const void *t1,
                         const void *s_over_den, const void *ratio, const float *h, const float *bias,
                         const void *gout, void *gx, void *gz, float *gh, float *gb, const void *taps,
                         void *workspace, size_t workspace_bytes, void *stream, float *pass_ms, bool gate = false)
{
    using namespace ndc;
    KGeom q;
    int st = make_kgeom(g, q);
    if (st) return st;
    q.gate = gate;
    if (!x || !z || !t1 || !h || !gout) return NDC_ERR_NULL;
    if ((s_over_den == nullptr) != (ratio == nullptr)) return NDC_ERR_NULL;
    if (!gx && !gz && !gh && !gb) return NDC_OK;
    const int path = choose_path(g, q);
    if (path < 0) return path;
    const size_t need = ndc_backward_workspace_bytes(g, gx != nullptr, gz != nullptr,
                                                     gh != nullptr, gb != nullptr);
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255u)))
        return NDC_ERR_WORKSPACE;
    if (path == NDC_PATH_FUSED) {
        const float *tp = fused::forward_ws(q, g->dtype) ? (const float *)taps : nullptr;
        return g->dtype == NDC_F32
                   ? fused::backward<Backend, float>(q, (const float *)x, (const float *)z,
                                                     (const float *)t1, (const float *)s_over_den,
                                                     (const float *)ratio, h, bias,
                                                     (const float *)gout, (float *)gx,
                                                     (float *)gz, gh, gb, tp, workspace, stream, pass_ms)
                   : fused::backward<Backend, bf16_t>(q, (const bf16_t *)x, (const bf16_t *)z,
                                                      (const bf16_t *)t1, (const bf16_t *)s_over_den,
                                                      (const bf16_t *)ratio, h, bias,
                                                      (const bf16_t *)gout, (bf16_t *)gx,
                                                      (bf16_t *)gz, gh, gb, tp, workspace, stream,
                                                      pass_ms);
    }
    return g->dtype == NDC_F32
               ? direct_backward<float>(q, (const float *)x, (const float *)z, (const float *)t1,
                                        h, bias, (const float *)gout, (float *)gx, (float *)gz,
                                        gh, gb, workspace, stream)
               : direct_backward<bf16_t>(q, (const bf16_t *)x, (const bf16_t *)z,
                                         (const bf16_t *)t1, h, bias, (const bf16_t *)gout,
                                         (bf16_t *)gx, (bf16_t *)gz, gh, gb, workspace, stream);
}

int ndc_backward(const ndc_geom *g, const void *x, const void *z, const void *t1,
                 const void *s_over_den, const void *ratio, const float *h, const float *bias,
                 const void *gout, void *gx, void *gz, float *gh, float *gb, void *workspace,
                 size_t workspace_bytes, void *stream)
{
    return backward_impl(g, x, z, t1, s_over_den, ratio, h, bias, gout, gx, gz, gh, gb, nullptr,
                         workspace, workspace_bytes, stream, nullptr);
}

int ndc_backward_taps(const ndc_geom *g, const void *x, const void *z, const void *t1,
                      const void *s_over_den, const void *ratio, const float *h, const void *taps,
                      const float *bias, const void *gout, void *gx, void *gz, float *gh, float *gb,
                      void *workspace, size_t workspace_bytes, void *stream)
{
    if (ndc_taps_bytes(g) && (!taps || ((uintptr_t)taps & 255u))) return NDC_ERR_WORKSPACE;
    return backward_impl(g, x, z, t1, s_over_den, ratio, h, bias, gout, gx, gz, gh, gb, taps,
                         workspace, workspace_bytes, stream, nullptr);
}

int ndc_backward_rectified(const ndc_geom *g, const void *x, const void *z, const void *t1,
                           const void *s_over_den, const void *ratio, const float *h, const void *taps,
                           const float *bias, const void *gout, void *gx, void *gz, float *gh, float *gb,
                           void *workspace, size_t workspace_bytes, void *stream)
{
    if (taps && ((uintptr_t)taps & 255u)) return NDC_ERR_WORKSPACE;
    return backward_impl(g, x, z, t1, s_over_den, ratio, h, bias, gout, gx, gz, gh, gb, taps,
                         workspace, workspace_bytes, stream, nullptr, true);
}

int ndc_backward_profiled(const ndc_geom *g, const void *x, const void *z, const void *t1,
                          const void *s_over_den, const void *ratio, const float *h,
                          const float *bias, const void *gout, void *gx, void *gz, float *gh,
                          float *gb, void *workspace, size_t workspace_bytes, void *stream,
                          float *pass_ms)
{
    if (!pass_ms) return NDC_ERR_NULL;
    pass_ms[0] = pass_ms[1] = pass_ms[2] = 0.f;
    return backward_impl(g, x, z, t1, s_over_den, ratio, h, bias, gout, gx, gz, gh, gb, nullptr,
                         workspace, workspace_bytes, stream, pass_ms);
}

int ndc_relayout(const void *src, void *dst, int64_t batch, int64_t channels, int64_t spatial,
                 int dtype, int to_channels_last, void *stream)
{
    if (!src || !dst) return NDC_ERR_NULL;
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || channels < 1 || spatial < 1 ||
        (long double)batch * channels * spatial > 9.0e15L)
        return NDC_ERR_GEOMETRY;
    if (src == dst) return NDC_ERR_GEOMETRY;
    // channels-last (B, S, C) -> channel-first (B, C, S) transposes S x C matrices, the other
    // direction C x S ones
    const long long R = to_channels_last ? channels : spatial, K = to_channels_last ? spatial : channels;
    const int st = ndc::Backend::transpose(src, dst, batch, R, K, dtype == NDC_BF16 ? 2 : 4, stream);
    return st == -2 ? (int)NDC_ERR_GEOMETRY : st;
}

// How a row of n elements is cut for the row normalisation: about 4096 workgroups in all, parts
// of at least 8192 elements and a multiple of 2048 (every thread's 16-byte vectors stay whole),
// at most 64 parts (one wavefront adds a row's partial sums).
static void rownorm_split(long long rows, long long n, int &nsplit, long long &chunk)
{
    long long want = (4096 + rows - 1) / rows;
    if (want > 64) want = 64;
    if (want > n / 8192) want = n / 8192;
    if (want < 1) want = 1;
    chunk = (n + want - 1) / want;
    chunk = (chunk + 2047) / 2048 * 2048;
    nsplit = (int)((n + chunk - 1) / chunk);
}

static int rownorm_check(long long rows, long long n, int dtype)
{
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (rows < 1 || n < 1 || (long double)rows * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    if (rows * nsplit > 0x7fffffffLL) return NDC_ERR_GEOMETRY;
    return NDC_OK;
}

size_t ndc_rownorm_workspace_bytes(int64_t rows, int64_t n)
{
    if (rows < 1 || n < 1) return 0;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    return (size_t)rows * nsplit * 2 * sizeof(float);
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

int ndc_rownorm_forward(const void *x, void *y, float *stats, int64_t rows, int64_t n, int dtype,
                        float eps, void *workspace, size_t workspace_bytes, void *stream)
{
    if (!x || !y || !stats || !workspace) return NDC_ERR_NULL;
    int st = rownorm_check(rows, n, dtype);
    if (st) return st;
    if (x == (const void *)y || !(eps >= 0.f)) return NDC_ERR_GEOMETRY;
    if (workspace_bytes < ndc_rownorm_workspace_bytes(rows, n) || ((uintptr_t)workspace & 7u))
        return NDC_ERR_WORKSPACE;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(x) && aligned16(y);
    return ndc::Backend::rownorm(false, x, nullptr, nullptr, (float *)workspace, stats, y, rows, n, nsplit,
                                 chunk, esz, vec, eps, stream);
}

int ndc_rownorm_stats(const void *x, float *stats, int64_t rows, int64_t n, int dtype, float eps, void *workspace,
                      size_t workspace_bytes, void *stream)
{
    if (!x || !stats || !workspace) return NDC_ERR_NULL;
    const int st = rownorm_check(rows, n, dtype);
    if (st) return st;
    if (!(eps >= 0.f)) return NDC_ERR_GEOMETRY;
    if (workspace_bytes < ndc_rownorm_workspace_bytes(rows, n) || ((uintptr_t)workspace & 7u) || ((uintptr_t)stats & 7u))
        return NDC_ERR_WORKSPACE;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(x);
    return ndc::Backend::rownorm_stats(x, (float *)workspace, stats, rows, n, nsplit, chunk, esz, vec, eps, stream);
}

int ndc_rownorm_backward(const void *gy, const void *y, const float *stats, const void *addend, void *gx,
                         int64_t rows, int64_t n, int dtype, void *workspace, size_t workspace_bytes,
                         void *stream)
{
    if (!gy || !y || !stats || !gx || !workspace) return NDC_ERR_NULL;
    int st = rownorm_check(rows, n, dtype);
    if (st) return st;
    if (gx == y) return NDC_ERR_GEOMETRY;
    if (workspace_bytes < ndc_rownorm_workspace_bytes(rows, n) || ((uintptr_t)workspace & 7u))
        return NDC_ERR_WORKSPACE;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(gy) && aligned16(y) && aligned16(gx) &&
                     (!addend || aligned16(addend));
    return ndc::Backend::rownorm(true, gy, y, addend, (float *)workspace, const_cast<float *>(stats), gx, rows,
                                 n, nsplit, chunk, esz, vec, 0.f, stream);
}

static int bias_act_check(long long batch, long long channels, long long n, int act, int dtype)
{
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || channels < 1 || channels > 0x7fffffffLL || n < 1 || act < NDC_ACT_NONE || act > NDC_ACT_GELU)
        return NDC_ERR_GEOMETRY;
    if ((long double)batch * channels * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    return rownorm_check(batch * channels, n, dtype);
}

int64_t ndc_bias_act_parts(int64_t rows, int64_t n)
{
    if (rows < 1 || n < 1) return 0;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    return nsplit;
}

int ndc_bias_act(const void *z, const float *bias, const void *residual, void *y, int64_t batch,
                 int64_t channels, int64_t n, int act, int dtype, void *stream)
{
    if (!z || !y) return NDC_ERR_NULL;
    int st = bias_act_check(batch, channels, n, act, dtype);
    if (st) return st;
    int nsplit;
    long long chunk;
    rownorm_split(batch * channels, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(z) && aligned16(y) && (!residual || aligned16(residual));
    return ndc::Backend::bias_act(z, bias, residual, y, batch * channels, (int)channels, n, nsplit, chunk, act,
                                  esz, vec, stream);
}

int ndc_bias_act_backward(const void *gy, const void *z, const float *bias, void *gz, float *gpart,
                          int64_t batch, int64_t channels, int64_t n, int act, int dtype, void *stream)
{
    if (!gy || !z || !gz) return NDC_ERR_NULL;
    int st = bias_act_check(batch, channels, n, act, dtype);
    if (st) return st;
    if (act == NDC_ACT_NONE) return NDC_ERR_GEOMETRY;   // gz = gy: nothing to compute
    int nsplit;
    long long chunk;
    rownorm_split(batch * channels, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(gy) && aligned16(z) && aligned16(gz);
    return ndc::Backend::bias_act_backward(gy, z, bias, gz, gpart, batch * channels, (int)channels, n, nsplit,
                                           chunk, act, esz, vec, stream);
}

// ---- streaming GEMM of the 1x1 projections (ndc_pwgemm.h)

int ndc_pointwise_gemm_supported(int64_t cin, int64_t cout, int64_t n, int dtype)
{
    if (dtype != NDC_BF16) return 0;
    // up to 256 input channels held whole in registers, any width of output; or many input
    // channels in chunks of 64 with the accumulators of at most 128 output channels
    const bool whole = cin == 32 || cin == 64 || cin == 128 || cin == 256;
    const bool deep = cin > 256 && cin % 64 == 0 && cin <= 4096 && cout <= 128;
    if (!whole && !deep) return 0;
    if (cout < 32 || cout % 32 || cout > 4096) return 0;
    if (cin * cout * 2 > 128 * 1024) return 0;        // the packed weights stay in LDS,
    if (cin * cout * 2 + cout * 36 > 160 * 1024) return 0;   // with the bias and eight rows of sums
    if (n < 64 || n % 64) return 0;
    return 1;
}

size_t ndc_pointwise_weight_bytes(int64_t cin, int64_t cout)
{
    return cin > 0 && cout > 0 ? (size_t)cin * (size_t)cout * 2 : 0;
}

int ndc_pointwise_pack(const void *w, int w_dtype, int transposed, void *wfrag, int64_t cin, int64_t cout,
                       void *stream)
{
    if (!w || !wfrag) return NDC_ERR_NULL;
    if (w_dtype != NDC_F32 && w_dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (cin < 16 || cin % 16 || cout < 32 || cout % 32 || cin > 4096 || cout > 4096) return NDC_ERR_GEOMETRY;
    if ((uintptr_t)wfrag & 15u) return NDC_ERR_WORKSPACE;
    return ndc::Backend::pwgemm_pack(w, w_dtype == NDC_BF16, transposed != 0, wfrag, (int)cout, (int)cin, stream);
}

int ndc_pointwise_gemm(const void *x, const void *wfrag, const float *bias, const void *residual, void *y,
                       void *zkeep, int64_t batch, int64_t cin, int64_t cout, int64_t n, int act, int dtype,
                       void *stream)
{
    if (!x || !wfrag || !y) return NDC_ERR_NULL;
    if (dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || act < NDC_ACT_NONE || act > NDC_ACT_GELU) return NDC_ERR_GEOMETRY;
    if (!ndc_pointwise_gemm_supported(cin, cout, n, dtype)) return NDC_ERR_GEOMETRY;
    if ((long double)batch * (cin > cout ? cin : cout) * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    if (batch * (n / 64) > 0x7fffff00LL || n > 0x3fffffffLL) return NDC_ERR_GEOMETRY;   // 32-bit tile count and lane offsets
    // word accesses on voxel pairs, 16-byte reads of the weights
    if (((uintptr_t)x & 3u) || ((uintptr_t)y & 3u) || (residual && ((uintptr_t)residual & 3u)) ||
        (zkeep && ((uintptr_t)zkeep & 3u)) || ((uintptr_t)wfrag & 15u) || (bias && ((uintptr_t)bias & 3u)))
        return NDC_ERR_WORKSPACE;
    if (y == x || zkeep == x || (zkeep && zkeep == y)) return NDC_ERR_GEOMETRY;
    if (cin > 256 && (act != NDC_ACT_NONE || zkeep)) return NDC_ERR_GEOMETRY;   // see the header
    if (act == NDC_ACT_NONE && zkeep) return NDC_ERR_GEOMETRY;   // without an activation y - bias is the product
    return ndc::Backend::pwgemm(x, wfrag, bias, residual, y, zkeep, nullptr, nullptr, batch, (int)cin, (int)cout, n, act,
                                stream);
}

int ndc_pointwise_gemm_normed_supported(int64_t cin, int64_t cout, int64_t n, int act)
{
    const bool square = act == NDC_ACT_RELU && cin == cout && (cin == 32 || cin == 64 || cin == 128);
    const bool hidden = act == NDC_ACT_GELU && cin == 128 && cout == 512;
    return (square || hidden) && ndc_pointwise_gemm_supported(cin, cout, n, NDC_BF16);
}

int ndc_pointwise_gemm_normed(const void *x, const float *stats, const void *wfrag, const float *bias, void *y, int64_t batch,
                              int64_t cin, int64_t cout, int64_t n, int act, int dtype, void *stream)
{
    if (!x || !stats || !wfrag || !y) return NDC_ERR_NULL;
    if (dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || !ndc_pointwise_gemm_normed_supported(cin, cout, n, act)) return NDC_ERR_GEOMETRY;
    if ((long double)batch * cout * n > 9.0e15L || batch * (n / 64) > 0x7fffff00LL || n > 0x3fffffffLL) return NDC_ERR_GEOMETRY;
    if (((uintptr_t)x & 3u) || ((uintptr_t)y & 3u) || ((uintptr_t)wfrag & 15u) || ((uintptr_t)bias & 3u) || ((uintptr_t)stats & 15u))
        return NDC_ERR_WORKSPACE;
    if (y == x) return NDC_ERR_GEOMETRY;
    return ndc::Backend::pwgemm_normed(x, stats, wfrag, bias, y, batch, (int)cin, (int)cout, n, act, stream);
}

int ndc_pointwise_gemm_masked(const void *x, const void *wfrag, const float *bias, const void *residual,
                              const void *mask, void *y, int64_t batch, int64_t cin, int64_t cout, int64_t n,
                              int dtype, void *stream)
{
    if (!x || !wfrag || !y || !mask) return NDC_ERR_NULL;
    if (dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || !ndc_pointwise_gemm_supported(cin, cout, n, dtype)) return NDC_ERR_GEOMETRY;
    if ((long double)batch * (cin > cout ? cin : cout) * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    if (batch * (n / 64) > 0x7fffff00LL || n > 0x3fffffffLL) return NDC_ERR_GEOMETRY;
    if (((uintptr_t)x & 3u) || ((uintptr_t)y & 3u) || ((uintptr_t)mask & 3u) || (residual && ((uintptr_t)residual & 3u)) ||
        ((uintptr_t)wfrag & 15u) || (bias && ((uintptr_t)bias & 3u)))
        return NDC_ERR_WORKSPACE;
    if (y == x || y == mask) return NDC_ERR_GEOMETRY;
    return ndc::Backend::pwgemm(x, wfrag, bias, residual, y, nullptr, nullptr, mask, batch, (int)cin, (int)cout, n, 5, stream);
}

int64_t ndc_pointwise_gemm_parts(void)
{
    return 4096;
}

int ndc_pointwise_gemm_actgrad(const void *gy, const void *wfrag, const float *bias, const void *z, void *gz,
                               float *gpart, int64_t batch, int64_t cin, int64_t cout, int64_t n, int act,
                               int dtype, void *stream)
{
    if (!gy || !wfrag || !z || !gz) return NDC_ERR_NULL;
    if (dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || (act != NDC_ACT_RELU && act != NDC_ACT_GELU)) return NDC_ERR_GEOMETRY;
    if (!ndc_pointwise_gemm_supported(cin, cout, n, dtype) || cin > 256) return NDC_ERR_GEOMETRY;
    if ((long double)batch * (cin > cout ? cin : cout) * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    if (batch * (n / 64) > 0x7fffff00LL || n > 0x3fffffffLL) return NDC_ERR_GEOMETRY;
    if (((uintptr_t)gy & 3u) || ((uintptr_t)gz & 3u) || ((uintptr_t)z & 3u) || ((uintptr_t)wfrag & 15u) ||
        (bias && ((uintptr_t)bias & 3u)) || (gpart && ((uintptr_t)gpart & 3u)))
        return NDC_ERR_WORKSPACE;
    if (gz == gy || gz == z) return NDC_ERR_GEOMETRY;
    return ndc::Backend::pwgemm(gy, wfrag, bias, z, gz, nullptr, gpart, nullptr, batch, (int)cin, (int)cout, n, act + 2, stream);
}

// ---- the MLP with its hidden tensor on chip (ndc_mlp.h)

int ndc_mlp_supported(int64_t c, int64_t n, int dtype)
{
    return dtype == NDC_BF16 && (c == 32 || c == 64) && n >= 64 && n % 64 == 0 && n <= (1LL << 26);
}

static int mlp_check(int64_t batch, int64_t c, int64_t n, int w_dtype, int dtype)
{
    if (dtype != NDC_BF16 || (w_dtype != NDC_F32 && w_dtype != NDC_BF16)) return NDC_ERR_DTYPE;
    if (batch < 1 || !ndc_mlp_supported(c, n, dtype) || (long double)batch * n > 64.0L * 0x7fffff00LL) return NDC_ERR_GEOMETRY;
    return NDC_OK;
}

int ndc_mlp_forward(const void *x, const float *stats, const void *w1, const void *w2, int w_dtype, const float *b1, const float *b2,
                    const void *residual, void *y, int64_t batch, int64_t c, int64_t n, int dtype, void *stream)
{
    if (!x || !w1 || !w2 || !y || (stats && !residual)) return NDC_ERR_NULL;
    if ((uintptr_t)stats & 15u) return NDC_ERR_WORKSPACE;
    const int st = mlp_check(batch, c, n, w_dtype, dtype);
    if (st) return st;
    // (weights are loaded element by element)
    const uintptr_t wmask = w_dtype == NDC_BF16 ? 1u : 3u;
    if (((uintptr_t)x & 3u) || ((uintptr_t)y & 3u) || ((uintptr_t)residual & 3u) || ((uintptr_t)b1 & 3u) || ((uintptr_t)b2 & 3u) ||
        ((uintptr_t)w1 & wmask) || ((uintptr_t)w2 & wmask))
        return NDC_ERR_WORKSPACE;
    if (y == x) return NDC_ERR_GEOMETRY;
    return ndc::Backend::mlp_forward(x, stats, w1, w2, w_dtype == NDC_BF16, b1, b2, residual, y, batch, (int)c, n, stream);
}

size_t ndc_mlp_workspace_bytes(int64_t batch, int64_t c, int64_t n)
{
    if (batch < 1 || !ndc_mlp_supported(c, n, NDC_BF16)) return 0;
    return (size_t)ndc::mlp::grad_groups(batch * (n / 64)) * (size_t)ndc::mlp::part_floats((int)c) * 4;
}

int ndc_mlp_backward(const void *x, const void *gy, const void *w1, const void *w2, int w_dtype, const float *b1,
                     void *gx, float *gw1, float *gb1, float *gw2, float *gb2, int64_t batch, int64_t c, int64_t n,
                     int dtype, void *workspace, size_t workspace_bytes, void *stream)
{
    if (!x || !gy || !w1 || !w2) return NDC_ERR_NULL;
    const int st = mlp_check(batch, c, n, w_dtype, dtype);
    if (st) return st;
    const uintptr_t wmask = w_dtype == NDC_BF16 ? 1u : 3u;
    if (((uintptr_t)x & 15u) || ((uintptr_t)gy & 15u) || ((uintptr_t)gx & 3u) || ((uintptr_t)b1 & 3u) || ((uintptr_t)w1 & wmask) ||
        ((uintptr_t)w2 & wmask) || !workspace || ((uintptr_t)workspace & 15u) || workspace_bytes < ndc_mlp_workspace_bytes(batch, c, n))
        return NDC_ERR_WORKSPACE;
    if (gx == x || gx == gy) return NDC_ERR_GEOMETRY;
    if (!gx && !gw1 && !gb1 && !gw2 && !gb2) return NDC_OK;
    return ndc::Backend::mlp_backward(x, gy, w1, w2, w_dtype == NDC_BF16, b1, gx, gw1, gb1, gw2, gb2, (float *)workspace, batch, (int)c,
                                      n, stream);
}

// ---- training loss (ndc_loss.h)

// Parts of a row, a workgroup each: about 2048 in all where a part keeps 2048 elements, and a part has at
// most 65536 (a thread then sums 256 terms).  One workgroup adds the parts of all rows, a wavefront a row:
// that is sized for some hundred rows, hence the limit.
static int dice_split(long long rows, long long n, int &parts, long long &chunk)
{
    if (rows < 1 || n < 1 || rows > 1024 || n > (1LL << 36)) return NDC_ERR_GEOMETRY;
    long long want = (2048 + rows - 1) / rows;
    if (want > n / 2048) want = n / 2048;
    if (want < (n + 65535) / 65536) want = (n + 65535) / 65536;
    chunk = (n + want - 1) / want;
    parts = (int)((n + chunk - 1) / chunk);
    return rows * parts < (1LL << 31) ? NDC_OK : NDC_ERR_GEOMETRY;
}

size_t ndc_dice_bce_workspace_bytes(int64_t rows, int64_t n)
{
    int parts;
    long long chunk;
    return dice_split(rows, n, parts, chunk) ? 0 : (size_t)rows * parts * 16;
}

int ndc_dice_bce_forward(const float *logits, const float *target, float *loss, float *coef, int64_t rows, int64_t n,
                         void *workspace, size_t workspace_bytes, void *stream)
{
    if (!logits || !target || !loss || !coef || !workspace) return NDC_ERR_NULL;
    int parts;
    long long chunk;
    const int st = dice_split(rows, n, parts, chunk);
    if (st) return st;
    if (workspace_bytes < (size_t)rows * parts * 16 || ((uintptr_t)workspace & 15u) || ((uintptr_t)coef & 7u)) return NDC_ERR_WORKSPACE;
    return ndc::Backend::dice_bce_forward(logits, target, loss, coef, (float *)workspace, (int)rows, n, parts, chunk, stream);
}

int ndc_dice_bce_backward(const float *logits, const float *target, const float *coef, const float *gloss,
                          float *glogits, int64_t rows, int64_t n, void *stream)
{
    if (!logits || !target || !coef || !gloss || !glogits) return NDC_ERR_NULL;
    int parts;
    long long chunk;
    const int st = dice_split(rows, n, parts, chunk);
    if (st) return st;
    if ((uintptr_t)coef & 7u) return NDC_ERR_WORKSPACE;
    return ndc::Backend::dice_bce_backward(logits, target, coef, gloss, glogits, (int)rows, n, parts, chunk, stream);
}

// ---- optimiser step (ndc_adamw.h)

int ndc_adamw(const ndc_adamw_tensor *tensors, int64_t count, double lr, double beta1, double beta2, double eps,
              double weight_decay, void *stream)
{
    if (count < 0 || count > (1 << 24)) return NDC_ERR_GEOMETRY;
    if (count && !tensors) return NDC_ERR_NULL;
    for (int64_t i = 0; i < count; ++i) {
        const ndc_adamw_tensor &t = tensors[i];
        if (t.n < 0 || t.n > (1LL << 40)) return NDC_ERR_GEOMETRY;
        if (!t.step || (t.n && (!t.param || !t.grad || !t.m || !t.v))) return NDC_ERR_NULL;
        if (((uintptr_t)t.param | (uintptr_t)t.grad | (uintptr_t)t.m | (uintptr_t)t.v | (uintptr_t)t.step) & 3u) return NDC_ERR_WORKSPACE;
    }
    if (!count) return NDC_OK;
    return ndc::Backend::adamw(tensors, count, lr, beta1, beta2, eps, weight_decay, stream);
}

// ---- the tiled GEMMs (ndc_gemm.h)

static int gemm_check(long long batch, long long cin, long long cout, long long n, int dtype)
{
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (batch < 1 || cin < 1 || cout < 1 || n < 1 || cin > (1 << 20) || cout > (1 << 20) || batch > (1 << 20)) return NDC_ERR_GEOMETRY;
    if ((long double)batch * (cin > cout ? cin : cout) * n > 9.0e15L || n > (1 << 24)) return NDC_ERR_GEOMETRY;
    return NDC_OK;
}

// Tile and split of a weight gradient.  The tile holds as much of the result as one workgroup's
// registers take (each operand is read once per tile that shares it), unless the voxels are too
// few to give 256 such tiles and splits, where 64 x 64 tiles spread the work wider.  The voxel
// axis is split until the launch has 512 workgroups (256 with the largest tiles over long rows:
// 0.55 ms against 0.56-0.68 for the 256 x 64 result over 2 x 128^3), in chunks of at least 256 voxels,
// so that partial results stay small next to the operands; of at least 64 where that leaves CUs
// without a workgroup, whose stages each wait for memory (128 x 32 over 16 384 voxels in float32, 64
// splits, 9.8 us, 256 of them 6.0).  Rows of half a million voxels and
// more are read 16 granules at a time (see the kernel), shorter ones 8.
static ndc::WgradPlan wgrad_plan(long long batch, long long rows, long long cols, long long n, int esz)
{
    ndc::WgradPlan w;
    if (rows >= 192 && cols <= 64) w.bm = 256, w.bn = 64;
    else if (cols >= 192 && rows <= 64) w.bm = 64, w.bn = 256;
    else if (rows > 64 && cols > 64) w.bm = w.bn = 128;
    else if (cols <= 32 && rows > 64) w.bm = 128, w.bn = 32;
    else if (rows <= 32 && cols > 64) w.bm = 32, w.bn = 128;
    else w.bm = w.bn = 64;
    long long most = n / 256 > 0 ? n / 256 : 1;                   // splits of a sample
    auto tiles_of = [&] { return ((rows + w.bm - 1) / w.bm) * ((cols + w.bn - 1) / w.bn); };
    // (lane offsets within a tile are 32-bit: fewer rows per tile on enormous grids)
    if (tiles_of() * most * batch < 256 || (long double)(w.bm > w.bn ? w.bm : w.bn) * n * esz > 4.0e9L) w.bm = w.bn = 64;
    w.depth = esz == 2 && n >= (1 << 19) ? 16 : 8;
    const long long stage = 16 / esz * w.depth, tiles = tiles_of();   // voxels per stage
    const long long want = w.bm + w.bn == 320 && n >= (1 << 19) ? 256 : 512;
    if (tiles * most * batch < 256 && n >= 128) most = n / 64;
    long long per = (want + tiles * batch - 1) / (tiles * batch);
    if (per > most) per = most;
    if (esz == 4 && per < n / 2048) per = n / 2048;   // (the error of a split's chain of sums: 2^15 voxels 1.3 times the float32 instruction's)
    w.chunk = ((n + per - 1) / per + stage - 1) / stage * stage;
    w.per_sample = (int)((n + w.chunk - 1) / w.chunk);
    // Few voxels: no splits (per_sample 0, see wgrad_whole_kernel).  us, this and the split form with its
    // sum, float32 / bf16: 64 x 64 over 256 voxels 6.4 -> 3.6 / 5.4 -> 3.1, over 1024 6.5 -> 6.2 / 5.7 -> 4.4,
    // over 2048 7.2 -> 9.6 / 6.3 -> 6.1; 512 x 512 over 512 in tiles of 32 13.4 -> 6.7 / 11.7 -> 4.7 (in tiles
    // of 16 10.7 / 7.4).  Rows that end within 16 bytes read their last turns element by element: 512 x 512
    // over 500 13.0 -> 7.0 / 10.8 -> 4.3, 64 x 64 over 3 x 343 7.1 -> 4.9 / 8.6 -> 9.8.  More than 16 samples
    // spread over the chip by themselves unless the result is large: with the projection itself, over 64 x 16
    // voxels, 32 x 32 in bf16 10.5 -> 21, 256 x 256 28.5 -> 14.8 / 26.3 -> 23.9, 512 x 512 64 -> 38 / 54 -> 18.
    const bool ragged = n * esz % 16 != 0;
    if (batch * w.per_sample > 1 && batch * n <= (ragged ? 512 : 1024) && (batch <= 16 || rows * cols >= 64 * 1024)) {
        w.per_sample = 0, w.bm = w.bn = 16;
        if (tiles_of() > 256) w.bm = w.bn = 32;
    }
    return w;
}

size_t ndc_weight_grad_workspace_bytes(int64_t batch, int64_t rows, int64_t cols, int64_t n, int dtype)
{
    if (gemm_check(batch, cols, rows, n, dtype)) return 0;
    const ndc::WgradPlan w = wgrad_plan(batch, rows, cols, n, dtype == NDC_BF16 ? 2 : 4);
    const long long splits = batch * w.per_sample;
    return splits <= 1 ? 0 : (size_t)splits * (size_t)(rows * cols + rows) * 4;
}

int ndc_weight_grad(const void *gz, const void *x, float *gw, float *gb, int64_t batch, int64_t rows, int64_t cols,
                    int64_t n, int dtype, void *workspace, size_t workspace_bytes, void *stream)
{
    if (!gz || !x || !gw) return NDC_ERR_NULL;
    int st = gemm_check(batch, cols, rows, n, dtype);
    if (st) return st;
    const size_t need = ndc_weight_grad_workspace_bytes(batch, rows, cols, n, dtype);
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15u))) return NDC_ERR_WORKSPACE;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    if (((uintptr_t)gz | (uintptr_t)x) & (uintptr_t)(esz - 1)) return NDC_ERR_WORKSPACE;
    const ndc::WgradPlan w = wgrad_plan(batch, rows, cols, n, esz);
    const long long splits = batch * w.per_sample, out = rows * cols;
    const long long blocks = ((splits + 7) / 8 * 8) * ((rows + w.bm - 1) / w.bm) * ((cols + w.bn - 1) / w.bn);
    if (blocks > 0x7fffffffLL || out + rows > 0x7fffffffLL) return NDC_ERR_GEOMETRY;
    float *part = need ? (float *)workspace : nullptr;
    st = ndc::Backend::wgrad(gz, x, gw, gb, part, batch, (int)rows, (int)cols, n, esz, w, stream);
    if (st || !part) return st;
    const int total = (int)(out + (gb ? rows : 0)), nout = (int)out;
    const long long stride = out + rows;
    return ndc::Backend::strided_sum(total, (int)splits, stream,
                                     [=] NDC_LAMBDA(int o, float v) { if (o < nout) gw[o] = v; else gb[o - nout] = v; },
                                     [=] NDC_LAMBDA(int o, int s) { return part[s * stride + o]; });
}

// How ndc_gemm cuts its work: blocks of 32 output rows that a workgroup makes of a 128-voxel tile, or
// one of the small-grid forms, which slice the channels over the wavefronts (waves <= 0), in tiles of 32
// rows x 64 voxels or (-1) of 16 rows x 32 voxels: in float32 the smaller ones while they are at most two per CU (us,
// 512 -> 128 channels over 1000 voxels, 64 of the larger tiles, 5.7 against 9.4; over 2288, 144 of them, 11.3 against
// 9.9; 1024 -> 256 over 8 x 256, 256 of them, 25 against 18).
// bf16 is sliced up to four workgroups per CU (128 -> 512 channels over 4096 voxels 8.1 us against 10.2 tiled,
// over 32 768, 4096 workgroups, 24 against 11.5), in the smaller tiles up to four of those per CU (512 -> 128 over 1000
// 4.8 against 5.6; past two they are behind, 7.2 against 5.7 over 2288, but the two forms add the channels in another
// order, and results that are rounded to bf16 keep their bits where the line is).  Otherwise as many output rows per
// workgroup (32 per wavefront) as still leave two workgroups per CU.
// float32 is sliced up to 600 workgroups (us, sliced / tiled: 512 -> 2048 over 572, 576 of them, 22.1 / 23.1, 512 -> 512
// over 8 x 256, 512, 17.1 / 17.9; 1024 -> 256 over 2 x 3375, 848, 55 / 43; 256 -> 256 over 8 x 1024, 1024, 19 / 13.7).
// Samples that fill half of a tile or less are sliced, as bf16 is, up to 1024 workgroups and in the smaller tiles up to 256
// of the larger ones (us, sliced / tiled: 1024 -> 256 over 96 x 4, 768 of them, 39 / 56, over 90 x 32 40 / 56; 256 -> 256 over
// 96 x 16 13.6 / 18.6; 512 -> 128 over 179 x 64 25 / 33; smaller tiles / larger: 1024 -> 256 over 20 x 2, 160, 12.8 / 15.2).
// Otherwise 64 rows a workgroup from 400 of those on (256 -> 256 over 13 824, 432 of them, 19 against 21 with 32 rows;
// 512 -> 128 over 20 000, 314, 31 against 29).
static int gemm_waves(long long batch, long long cin, long long cout, long long n, int esz)
{
    const long long vt = batch * ((n + 127) / 128), small = batch * ((n + 63) / 64) * ((cout + 31) / 32);
    if (small <= (esz == 4 && n > 64 ? 600 : 1024) && cin % (16 / esz) == 0 && n >= 2)
        return small <= (esz == 4 && n > 32 ? 128 : 256) ? -1 : 0;
    if (esz == 4) return cout > 32 && vt * ((cout + 63) / 64) >= 400 ? 2 : 1;
    int waves = 4;
    while (waves > 1 && (cout <= 32 * (waves / 2) || vt * ((cout + 32 * waves - 1) / (32 * waves)) < 512)) waves /= 2;
    return waves;
}

// sizes that ndc_gemm takes
static int gemm_sizes(long long batch, long long cin, long long cout, long long n, int dtype)
{
    const int st = gemm_check(batch, cin, cout, n, dtype);
    if (st) return st;
    const long long vt = batch * ((n + 127) / 128);
    return (vt + 8) * 2 * ((cout + 31) / 32 + 8) > 0x7fffffffLL ? (int)NDC_ERR_GEOMETRY : (int)NDC_OK;
}

// voxels of a tile
static int gemm_tile(int waves) { return waves > 0 ? 128 : waves ? 32 : 64; }

static int gemm_impl(const void *x, const float *w, int transposed, const float *bias, const void *residual, const void *mask,
                     void *y, void *zkeep, float *gpart, int64_t batch, int64_t cin, int64_t cout, int64_t n, int mode,
                     int dtype, void *stream)
{
    if (!x || !w || !y) return NDC_ERR_NULL;
    const int st = gemm_sizes(batch, cin, cout, n, dtype);
    if (st) return st;
    if (mode < NDC_ACT_NONE || mode > NDC_GEMM_GELU_GRAD || mode == 3) return NDC_ERR_GEOMETRY;
    const bool grad = mode == NDC_GEMM_GELU_GRAD, act = mode == NDC_ACT_RELU || mode == NDC_ACT_GELU;
    if (grad && !residual) return NDC_ERR_NULL;
    if (mask && mode != NDC_ACT_NONE) return NDC_ERR_GEOMETRY;
    if (zkeep && !act) return NDC_ERR_GEOMETRY;
    if ((act && transposed) || (grad && !transposed)) return NDC_ERR_GEOMETRY;   // forms no caller has
    const uintptr_t all = (uintptr_t)x | (uintptr_t)y | (uintptr_t)residual | (uintptr_t)mask | (uintptr_t)zkeep;
    if (all & (uintptr_t)((dtype == NDC_BF16 ? 2 : 4) - 1) || ((uintptr_t)w & 3u) || ((uintptr_t)bias & 3u) || ((uintptr_t)gpart & 3u))
        return NDC_ERR_WORKSPACE;
    if (y == x || zkeep == x || (zkeep && zkeep == y)) return NDC_ERR_GEOMETRY;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    return ndc::Backend::tile_gemm(x, w, transposed != 0, bias, residual, mask, y, zkeep, gpart, batch, (int)cin, (int)cout, n,
                                   mode, esz, gemm_waves(batch, cin, cout, n, esz), stream);
}

int ndc_gemm(const void *x, const float *w, int transposed, const float *bias, const void *residual, const void *mask,
             void *y, void *zkeep, int64_t batch, int64_t cin, int64_t cout, int64_t n, int mode, int dtype,
             void *stream)
{
    return gemm_impl(x, w, transposed, bias, residual, mask, y, zkeep, nullptr, batch, cin, cout, n, mode, dtype, stream);
}

int64_t ndc_gemm_parts(int64_t batch, int64_t cin, int64_t cout, int64_t n, int dtype)
{
    if (gemm_sizes(batch, cin, cout, n, dtype)) return 0;
    const int tile = gemm_tile(gemm_waves(batch, cin, cout, n, dtype == NDC_BF16 ? 2 : 4));
    return batch * ((n + tile - 1) / tile);
}

int ndc_gemm_gelu_grad(const void *gy, const float *w, const float *bias, const void *z, void *gz, float *gpart,
                       int64_t batch, int64_t cin, int64_t cout, int64_t n, int dtype, void *stream)
{
    return gemm_impl(gy, w, 1, bias, z, nullptr, gz, nullptr, gpart, batch, cin, cout, n, NDC_GEMM_GELU_GRAD, dtype, stream);
}

// Many rows are folded to 256 first, in place (a row r < 256 receives rows r, r + 256, ... and is read
// by its own sum only): one level has a workgroup per 32 columns, each with a round trip to memory per
// 64 rows.  256 columns on an MI355X, one level and two: 1024 rows 3.9 and 6.3 us, 2048 6.4 and 6.2,
// 4096 11.2 and 6.2 (32 and 1024 columns: the same within a microsecond).
int ndc_column_sums(float *partial, float *sums, int64_t rows, int64_t cols, void *stream)
{
    if (!partial || !sums) return NDC_ERR_NULL;
    if (rows < 1 || cols < 1 || cols > (1 << 22) || rows > 0x7fffffffLL) return NDC_ERR_GEOMETRY;
    if (rows > 2048) {
        const int nc = (int)cols, total = (int)rows;
        const int st = ndc::Backend::strided_sum(
            256 * nc, (total + 255) / 256, stream, [=] NDC_LAMBDA(int o, float v) { partial[o] = v; },
            [=] NDC_LAMBDA(int o, int s) {
                const int r = s * 256 + o / nc;
                return r < total ? partial[(long long)r * nc + o % nc] : 0.f;
            });
        if (st) return st;
        rows = 256;
    }
    const long long nc = cols;
    return ndc::Backend::strided_sum((int)cols, (int)rows, stream, [=] NDC_LAMBDA(int o, float v) { sums[o] = v; },
                                     [=] NDC_LAMBDA(int o, int s) { return partial[s * nc + o]; });
}

static int chnorm_check(long long B, long long C, long long n, int dtype)
{
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    if (B < 1 || C < 1 || C > 0x7fffffffLL || n < 1 || (long double)B * C * n > 9.0e15L) return NDC_ERR_GEOMETRY;
    return NDC_OK;
}

// 16-byte accesses (8 or 4 voxels per thread) where that still leaves a few hundred workgroups;
// on small grids one voxel per thread, so that the launch spreads over the chip
static bool chnorm_wide(long long batch, long long n, int esz)
{
    return n % (16 / esz) == 0 && batch * ndc::Backend::chnorm_blocks(n, esz, true) >= 256;
}

int64_t ndc_chnorm_parts(int64_t batch, int64_t n, int dtype)
{
    if (batch < 1 || n < 1 || (dtype != NDC_F32 && dtype != NDC_BF16)) return 0;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    // (the count for the access width the entry points use when the buffers are aligned; an
    // unaligned call where the wide form applies needs more rows and is refused)
    return batch * ndc::Backend::chnorm_blocks(n, esz, chnorm_wide(batch, n, esz)) * ndc::Backend::kChnormWaves;
}

int ndc_chnorm_forward(const void *x, const float *weight, const float *bias, void *y, float *stats,
                       int64_t batch, int64_t channels, int64_t n, int dtype, float eps, void *stream)
{
    if (!x || !y || !stats) return NDC_ERR_NULL;
    int st = chnorm_check(batch, channels, n, dtype);
    if (st) return st;
    if (x == (const void *)y || !(eps >= 0.f)) return NDC_ERR_GEOMETRY;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = chnorm_wide(batch, n, esz) && aligned16(x) && aligned16(y);
    st = ndc::Backend::chnorm(false, nullptr, x, stats, weight, bias, y, nullptr, batch, (int)channels, n, esz, vec,
                              ndc_chnorm_parts(batch, n, dtype), eps, stream);
    return st == -2 ? (int)NDC_ERR_GEOMETRY : st;
}

int ndc_chnorm_backward(const void *gy, const void *x, const float *stats, const float *weight, void *gx,
                        float *partial, int64_t batch, int64_t channels, int64_t n, int dtype, void *stream)
{
    if (!gy || !x || !stats || !gx) return NDC_ERR_NULL;
    int st = chnorm_check(batch, channels, n, dtype);
    if (st) return st;
    if (gx == x) return NDC_ERR_GEOMETRY;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool fits = chnorm_wide(batch, n, esz);
    const bool vec = fits && aligned16(gy) && aligned16(x) && aligned16(gx);
    // the partial rows are laid out for the path ndc_chnorm_parts counted
    if (partial && fits && !vec) return NDC_ERR_WORKSPACE;
    st = ndc::Backend::chnorm(true, gy, x, stats, weight, nullptr, gx, partial, batch, (int)channels, n, esz, vec,
                              ndc_chnorm_parts(batch, n, dtype), 0.f, stream);
    return st == -2 ? (int)NDC_ERR_GEOMETRY : st;
}

int ndc_row_sums(const void *x, float *partial, int64_t rows, int64_t n, int dtype, void *stream)
{
    if (!x || !partial) return NDC_ERR_NULL;
    int st = rownorm_check(rows, n, dtype);
    if (st) return st;
    int nsplit;
    long long chunk;
    rownorm_split(rows, n, nsplit, chunk);
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool vec = n % (16 / esz) == 0 && aligned16(x);
    return ndc::Backend::row_sums(x, partial, rows, n, nsplit, chunk, esz, vec, stream);
}

int ndc_regroup(const void *src, void *dst, const float *bias, int64_t rows, int64_t channels, int64_t D,
                 int64_t H, int64_t W, int depth2, int dtype, int to_channels, void *stream)
{
    if (!src || !dst) return NDC_ERR_NULL;
    if (dtype != NDC_F32 && dtype != NDC_BF16) return NDC_ERR_DTYPE;
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    if (rows < 1 || channels < 1 || D < 1 || H < 2 || W < 2 || D > 0x3fffffff || H > 0x3fffffff ||
        W > 0x3fffffff || channels > 0x7fffffff || (long double)rows * D * H * W > 9.0e15L)
        return NDC_ERR_GEOMETRY;
    // even windows, whole 16-byte vectors per row, aligned buffers; a bias only on the way back
    if (H % 2 || W % (16 / esz) || (depth2 && D % 2) || src == dst || !aligned16(src) || !aligned16(dst) ||
        (bias && to_channels))
        return NDC_ERR_GEOMETRY;
    const int st = ndc::Backend::regroup2(src, dst, bias, rows, (int)channels, (int)D, (int)H, (int)W,
                                          depth2 ? 1 : 0, esz, to_channels ? 1 : 0, stream);
    return st == -2 ? (int)NDC_ERR_GEOMETRY : st;
}

}  // extern "C"

template <typename E, int V>
static int columns_launch(const ndc::KGeom &q, const void *src, void *dst, long long rows, void *stream)
{
    const ndc::Columns<E, V> op = {q, (const E *)src, (E *)dst};
    return ndc::Backend::per_unit(rows * q.KT, q.SP / V, stream, op);
}

extern "C" {

int ndc_columns(const void *src, void *dst, int64_t rows, int64_t D, int64_t H, int64_t W, int kD, int kH, int kW,
                int dtype, void *stream)
{
    if (!src || !dst) return NDC_ERR_NULL;
    if (rows < 1 || rows > 0x7fffffffLL || D < 1 || H < 1 || W < 1 || D > 0x7fffffffLL || H > 0x7fffffffLL ||
        W > 0x7fffffffLL || (long double)D * H * W >= 2147483648.0L || src == dst)
        return NDC_ERR_GEOMETRY;
    const ndc_geom g = {(int)rows, 1, 1, 1, {(int)D, (int)H, (int)W}, {kD, kH, kW}, dtype, 0, NDC_PATH_DIRECT, 0.f};
    ndc::KGeom q;
    const int st = ndc::make_kgeom(&g, q);
    if (st) return st;
    if (rows * q.KT > 0x7fffffffLL) return NDC_ERR_GEOMETRY;
    // 16 bytes per store where rows are made of them
    const int esz = dtype == NDC_BF16 ? 2 : 4;
    const bool wide = W % (16 / esz) == 0 && aligned16(dst);
    int r;
    if (esz == 2) r = wide ? columns_launch<uint16_t, 8>(q, src, dst, rows, stream) : columns_launch<uint16_t, 1>(q, src, dst, rows, stream);
    else r = wide ? columns_launch<uint32_t, 4>(q, src, dst, rows, stream) : columns_launch<uint32_t, 1>(q, src, dst, rows, stream);
    return r == -2 ? (int)NDC_ERR_GEOMETRY : r;
}

int ndc_gconv(const ndc_geom *g, const void *in, const float *h, const float *bias, int adjoint,
              void *out, void *stream)
{
    using namespace ndc;
    KGeom q;
    int st = make_kgeom(g, q);
    if (st) return st;
    if (!in || !h || !out) return NDC_ERR_NULL;
    return g->dtype == NDC_F32
               ? direct_gconv<float, float>(q, (const float *)in, h, bias, adjoint, (float *)out,
                                            stream)
               : direct_gconv<bf16_t, bf16_t>(q, (const bf16_t *)in, h, bias, adjoint,
                                              (bf16_t *)out, stream);
}

}  // extern "C"
