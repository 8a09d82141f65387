// The autograd nodes of the package, natively: shape checks, output allocation, the calls into
// libdeconver_ndc.so and the backward formulas of the NDC update, the 1x1 projections, the MLP,
// the norms and the 2-tap regrouping (deconver/deconvolution/functional.py:97-207 and
// deconver/layers of the reference are what these nodes stand for).
//
// Why native: a step of these networks is some 600 kernel launches, and on small tensors it is
// bound by what the host does between them.  With the nodes written in Python (an autograd
// Function each, its operands marshalled through ctypes) a launch cost about 20 us of host time:
// a training step on one 32^3 volume took 12.7 ms for 5.7 ms of kernels, one forward + backward
// of a 32-channel 64^2 layer 0.48 ms for 0.15 ms of kernels.  The arithmetic stays behind the C
// ABI of include/deconver_ndc.h; nothing here computes on tensors except through it, the
// library GEMMs that choose_gemm leaves, and a few float32 sums of
// partial results.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_cpp_function.h>

#include "../../include/deconver_ndc.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------- helpers

void check(int status, const char *what)
{
    TORCH_CHECK(status == 0, what, " failed: ", ndc_status_string(status), " (status ", status, ")");
}

int dtype_tag(const Tensor &t)
{
    if (t.scalar_type() == at::kFloat) return NDC_F32;
    if (t.scalar_type() == at::kBFloat16) return NDC_BF16;
    TORCH_CHECK_TYPE(false, "NDC kernels store activations as float32 or bfloat16, got ", t.scalar_type());
}

// What every node works under: the device of its tensors current, autocast off (operands are
// already in the dtype the node computes in), and no autograd recording inside.
struct Scope {
    c10::OptionalDeviceGuard device;
    c10::impl::ExcludeDispatchKeyGuard autocast;
    at::AutoDispatchBelowADInplaceOrView below;
    void *stream;
    static c10::Device on_gpu(const Tensor &t)
    {
        TORCH_CHECK(t.is_cuda(), "the HIP kernels run on GPU tensors only");
        return t.device();
    }
    explicit Scope(const Tensor &t)
        : device(on_gpu(t)), autocast(c10::autocast_dispatch_keyset),
          stream((void *)c10::hip::getCurrentHIPStream(t.device().index()).stream())
    {
    }
};

const void *ptr(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void *out_ptr(const Tensor &t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
const float *fptr(const Tensor &t) { return (const float *)ptr(t); }
float *out_fptr(const Tensor &t) { return (float *)out_ptr(t); }

Tensor f32_vector(const OptTensor &t)
{
    if (!t || !t->defined()) return Tensor();
    return t->detach().to(at::kFloat).contiguous();
}

Tensor empty(at::IntArrayRef size, const Tensor &like) { return at::empty(size, like.options()); }
Tensor empty_f32(at::IntArrayRef size, const Tensor &like)
{
    return at::empty(size, like.options().dtype(at::kFloat));
}

// The kernels see pointers and the sizes of one tensor: what the others have to be is checked here,
// before anything is launched.
void check_device(const Tensor &t, const Tensor &like, const char *what)
{
    TORCH_CHECK(t.device() == like.device(), "expected all tensors on one device, but ", what, " is on ", t.device(),
                " and the input on ", like.device());
}

void check_vector(const OptTensor &t, const Tensor &like, int64_t entries, const char *what)
{
    if (!t || !t->defined()) return;
    check_device(*t, like, what);
    TORCH_CHECK_VALUE(t->numel() == entries, what, " has ", t->numel(), " entries, expected one per channel, ", entries);
}

// A 1x1 projection of `channels` channels over the voxels of x, (B, ., *S): its weight (rows of W,
// or with `transposed` of its transpose), bias and residual (B, cout, *S).  Returns cout.
int64_t check_projection(const Tensor &x, int64_t channels, const Tensor &w, bool transposed, const OptTensor &bias,
                         const OptTensor &res)
{
    TORCH_CHECK_VALUE(w.dim() >= 2, "expected a weight matrix, got ", w.sizes());
    const int64_t rows = w.size(0), cols = rows ? w.numel() / rows : 0, cout = transposed ? cols : rows;
    TORCH_CHECK((transposed ? rows : cols) == channels, "weight of shape ", w.sizes(), transposed ? " (transposed)" : "", " takes ",
                transposed ? rows : cols, " channels, but the input has ", channels);
    check_device(w, x, "the weight");
    check_vector(bias, x, cout, "the bias");
    if (res && res->defined()) {
        auto size = x.sizes().vec();
        size[1] = cout;
        TORCH_CHECK_VALUE(res->sizes() == at::IntArrayRef(size), "the residual has shape ", res->sizes(), ", expected ", size);
        check_device(*res, x, "the residual");
    }
    return cout;
}

// What comes back from a saved-tensor hook need not be what was saved: the tensor as the kernels read
// it, or an error.
Tensor check_saved(const Tensor &t, const Tensor &like, at::IntArrayRef size, at::ScalarType type)
{
    if (!t.defined()) return t;
    check_device(t, like, "a saved tensor");
    TORCH_CHECK_VALUE(t.scalar_type() == type && t.sizes() == size, "a saved tensor came back as ", t.scalar_type(), " ", t.sizes(),
                      ", expected ", type, " ", size);
    return t.contiguous();
}
Tensor check_saved(const Tensor &t, const Tensor &like) { return check_saved(t, like, like.sizes(), like.scalar_type()); }

bool wants_grad(const Tensor &t) { return t.defined() && t.requires_grad(); }
bool wants_grad(const OptTensor &t) { return t && wants_grad(*t); }

// The nodes have no forward-mode rule.  Where autograd records a call its engine says so; a call that
// it does not record would drop the tangents without a word.
void no_tangents() {}
template <class... Rest> void no_tangents(const Tensor &t, const Rest &...rest);
template <class... Rest> void no_tangents(const OptTensor &t, const Rest &...rest)
{
    no_tangents(t ? *t : Tensor(), rest...);
}
template <class... Rest> void no_tangents(const Tensor &t, const Rest &...rest)
{
    TORCH_CHECK(!t.defined() || !t._fw_grad(0).defined(), "the NDC nodes do not implement forward-mode differentiation");
    no_tangents(rest...);
}

// Which gradients the engine asks for, by forward argument.  (The engine counts only the
// arguments that are tensors.)
struct Needs {
    std::vector<int> edge;
    int count = 0;
    void arg(bool defined) { edge.push_back(defined ? count++ : -1); }
    std::vector<bool> ask(AutogradContext *ctx) const
    {
        std::vector<bool> out(edge.size());
        for (size_t i = 0; i < edge.size(); ++i) out[i] = edge[i] >= 0 && ctx->needs_input_grad(edge[i]);
        return out;
    }
};

// Gradients of a node that is differentiable once: under create_graph they come back attached
// to a node that refuses the second differentiation instead of silently dropping its terms.
variable_list once(variable_list grads, bool recording, const variable_list &gouts)
{
    if (!recording) return grads;
    bool any = false;
    for (auto &g : gouts) any = any || wants_grad(g);
    if (!any) return grads;
    auto err = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)grads.size());
    variable_list marked;
    for (auto &g : grads) marked.push_back(g.defined() ? g.detach().requires_grad_(true) : g);
    return (*err)(std::move(marked));
}

// ---------------------------------------------------------------------------- layouts

bool channels_last(const Tensor &t)
{
    if ((t.dim() != 4 && t.dim() != 5) || t.is_contiguous()) return false;
    return t.is_contiguous(t.dim() == 4 ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::ChannelsLast3d);
}

int64_t voxels(const Tensor &t)
{
    int64_t n = 1;
    for (int64_t d = 2; d < t.dim(); ++d) n *= t.size(d);
    return n;
}

Tensor channel_first(const Tensor &t, void *stream)
{
    if (t.is_contiguous()) return t;
    if (!channels_last(t)) return t.contiguous();
    Tensor out = empty(t.sizes(), t);
    check(ndc_relayout(ptr(t), out_ptr(out), t.size(0), t.size(1), voxels(t), dtype_tag(t), 0, stream), "ndc_relayout");
    return out;
}

Tensor to_channels_last(const Tensor &t, void *stream)
{
    Tensor out = at::empty(t.sizes(), t.options().memory_format(
                                          t.dim() == 4 ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::ChannelsLast3d));
    check(ndc_relayout(ptr(t), out_ptr(out), t.size(0), t.size(1), voxels(t), dtype_tag(t), 1, stream), "ndc_relayout");
    return out;
}

// ---------------------------------------------------------------------------- projections

// The matrix W (cout x cin) of a 1x1 projection as it lies in memory: rows of W, or rows of its
// transpose (a transposed convolution's weight).  Any floating dtype.
struct Matrix {
    Tensor m;
    bool transposed;
    Matrix(const Tensor &w, bool t) : m(w.detach()), transposed(t)
    {
        if (m.dim() != 2) m = m.reshape({m.size(0), -1});
        if (!m.is_contiguous()) m = m.contiguous();
    }
    int64_t cout() const { return m.size(transposed ? 1 : 0); }
    int64_t cin() const { return m.size(transposed ? 0 : 1); }
    // (rows of W, columns of W) as a dense operand of a library GEMM, in `dtype`
    Tensor dense(at::ScalarType dtype, bool transpose) const
    {
        Tensor w = m.to(dtype);
        return transpose != transposed ? w.t() : w;
    }
};

// the weight of a projection to `cout` channels as a backward finds it (see check_saved)
Matrix saved_weight(const Tensor &w, bool transposed, int64_t cout, const Tensor &like)
{
    check_device(w, like, "a saved weight");
    TORCH_CHECK_VALUE(w.dim() >= 2 && w.size(0) > 0, "a saved weight came back as ", w.sizes());
    const Matrix m(w, transposed);
    TORCH_CHECK_VALUE(m.cout() == cout, "a saved weight came back as ", w.sizes(), ", expected ", cout, " output channels");
    return m;
}

// Which GEMM makes a 1x1 projection (or an input gradient), by what was measured on an MI355X:
//   kStream   the streaming GEMM (ndc_pointwise_gemm): bf16 in its channel counts, from 2048 of its
//             64-voxel tiles on (below, filling its weight table costs more than the product: 128 ->
//             512 channels over 4096 voxels 45 us against 8 us tiled);
//   kTiled    the tiled GEMM (ndc_gemm): small products -- a library GEMM costs the host 15-19 us a
//             call, as much as the product --, and larger ones whose tail (bias, activation,
//             residual, mask) it takes along: float32 always, bf16 with at most 32 K weights (256
//             -> 1024 channels over 2 x 32^3 voxels: 85 us against 59 us by the library, which then
//             pays for one more pass over the result).  In float32 the larger ones without a tail too (us,
//             library / tiled: 64 -> 256 over 2 x 91 125 voxels 128 / 61, 256 -> 1024 over 2 x 27 000 277 / 212,
//             512 -> 128 over 8 x 4096 37.7 / 33.9, 128 -> 64 over 8 x 16 384 27.6 / 27.5), but for those from 1024
//             channels and more between 2 and 12 GFLOP (1024 -> 256 over 8 x 1024 36.9 / 42.2, 2048 -> 512 over
//             4 x 1000 65 / 82, over 8000, 17 GFLOP, 130 / 118), for samples that fill half a tile's 128 voxels or less
//             (256 -> 256 over 4197 x 4 130 / 446, over 1050 x 16 59 / 121, over 954 x 64 74 / 115, but over 210 x 80
//             45 / 39; 128 -> 512 over 1908 x 32 110 / 257; not up to 64 channels, 64 -> 64 over 8393 x 32 109 / 83), and
//             for sizes that the tiled GEMM refuses;
//   kLibrary  the rest.
enum Gemm { kStream, kTiled, kLibrary };

Gemm choose_gemm(const Tensor &x, int64_t cout, bool act_or_keep, bool tail)
{
    const int64_t B = x.size(0), cin = x.size(1), n = x.size(2);
    const bool half = x.scalar_type() == at::kBFloat16;
    const bool stream = half && !(cin > 256 && act_or_keep) && ndc_pointwise_gemm_supported(cin, cout, n, NDC_BF16);
    if (stream && B * n >= 2048 * 64) return kStream;
    if (n > (1 << 24)) return stream ? kStream : kLibrary;
    const double flops = 2.0 * (double)B * (double)n * (double)cin * (double)cout;
    if (!half) {
        const bool library = (cin >= 1024 && flops < 12e9) || (n <= 64 && cin * cout > 64 * 64) || !ndc_gemm_parts(B, cin, cout, n, NDC_F32);
        return !tail && flops >= 2e9 && library ? kLibrary : kTiled;
    }
    if (flops < 4e9) return kTiled;
    if (tail && cin * cout <= 32 * 1024) return kTiled;
    return stream ? kStream : kLibrary;
}

// W (or W^T) in the order the streaming GEMM reads it
Tensor pack(const Matrix &w, bool transpose, const Tensor &like, void *stream)
{
    Tensor m = w.m;
    if (m.scalar_type() != at::kFloat && m.scalar_type() != at::kBFloat16) m = m.to(at::kBFloat16);
    const int64_t cin = transpose ? w.cout() : w.cin(), cout = transpose ? w.cin() : w.cout();
    Tensor frag = at::empty({cin * cout}, like.options().dtype(at::kBFloat16));
    check(ndc_pointwise_pack(ptr(m), dtype_tag(m), transpose != w.transposed, out_ptr(frag), cin, cout, stream),
          "ndc_pointwise_pack");
    return frag;
}

Tensor batched(const Tensor &w, int64_t B) { return w.unsqueeze(0).expand({B, w.size(0), w.size(1)}); }

// y = epilogue(W x) or epilogue(W^T x) by the tiled GEMM
void tiled(const Matrix &w, bool transpose, const Tensor &x, const Tensor &bias, const Tensor &res, const Tensor &mask,
           const Tensor &y, const Tensor &z, int mode, void *stream)
{
    const Tensor m = w.m.scalar_type() == at::kFloat ? w.m : w.m.to(at::kFloat);
    check(ndc_gemm(ptr(x), fptr(m), transpose != w.transposed, fptr(bias), ptr(res), ptr(mask), out_ptr(y), out_ptr(z), x.size(0),
                   x.size(1), y.size(1), x.size(2), mode, dtype_tag(x), stream), "ndc_gemm");
}

// W x per sample
Tensor project(const Matrix &w, const Tensor &x, bool library, void *stream)
{
    const int64_t B = x.size(0), n = x.size(2), cout = w.cout();
    Tensor z = empty({B, cout, n}, x);
    const Gemm by = library ? kLibrary : choose_gemm(x, cout, false, false);
    if (by == kStream) {
        Tensor frag = pack(w, false, x, stream);
        check(ndc_pointwise_gemm(ptr(x), ptr(frag), nullptr, nullptr, out_ptr(z), nullptr, B, w.cin(), cout, n, NDC_ACT_NONE,
                                 NDC_BF16, stream), "ndc_pointwise_gemm");
    } else if (by == kTiled) {
        tiled(w, false, x, Tensor(), Tensor(), Tensor(), z, Tensor(), NDC_ACT_NONE, stream);
    } else {
        // one batched GEMM, the weight shared by the samples through a zero stride
        at::bmm_out(z, batched(w.dense(x.scalar_type(), false), B), x);
    }
    return z;
}

// W^T gz per sample, onto `accumulate` if given (which may be overwritten), zero where mask <= 0
Tensor project_back(const Matrix &w, const Tensor &gz, Tensor accumulate, const Tensor &mask, void *stream)
{
    const int64_t B = gz.size(0), n = gz.size(2), cin = w.cin(), cout = w.cout();
    if (cout == 1) {
        // an outer product, i.e. a broadcast multiplication at the memory rate (as a GEMM it ran
        // at a fifth of it)
        Tensor gx = at::mul(gz, w.m.reshape({1, -1, 1}).to(gz.scalar_type()));
        if (accumulate.defined()) gx = accumulate.add_(gx);
        return mask.defined() ? gx.mul_(mask.gt(0)) : gx;
    }
    const Gemm by = choose_gemm(gz, cin, false, accumulate.defined() || mask.defined());
    if (by == kLibrary) {
        Tensor wt = batched(w.dense(gz.scalar_type(), true), B), gx;
        if (accumulate.defined()) {
            gx = accumulate.baddbmm_(wt, gz);
        } else {
            gx = empty({B, cin, n}, gz);
            at::bmm_out(gx, wt, gz);
        }
        return mask.defined() ? gx.mul_(mask.gt(0)) : gx;
    }
    Tensor gx = empty({B, cin, n}, gz);
    if (by == kTiled) {
        tiled(w, true, gz, Tensor(), accumulate, mask, gx, Tensor(), NDC_ACT_NONE, stream);
        return gx;
    }
    Tensor frag = pack(w, true, gz, stream);
    if (mask.defined())
        check(ndc_pointwise_gemm_masked(ptr(gz), ptr(frag), nullptr, ptr(accumulate), ptr(mask), out_ptr(gx), B, cout, cin, n,
                                        NDC_BF16, stream), "ndc_pointwise_gemm_masked");
    else
        check(ndc_pointwise_gemm(ptr(gz), ptr(frag), nullptr, ptr(accumulate), out_ptr(gx), nullptr, B, cout, cin, n, NDC_ACT_NONE,
                                 NDC_BF16, stream), "ndc_pointwise_gemm");
    return gx;
}

// sum over batch and voxels, float32, one value per channel
Tensor channel_sums(const Tensor &g, void *stream)
{
    const int64_t B = g.size(0), C = g.size(1), n = g.size(2);
    const int64_t parts = ndc_bias_act_parts(B * C, n);
    Tensor partial = empty_f32({B, C, parts}, g);
    check(ndc_row_sums(ptr(g), out_fptr(partial), B * C, n, dtype_tag(g), stream), "ndc_row_sums");
    return partial.sum(at::IntArrayRef{0, 2});
}

// sum over the rows of float32 partial results (rows, channels), which are overwritten
Tensor column_sums(const Tensor &partial, void *stream)
{
    Tensor sums = empty_f32({partial.size(1)}, partial);
    check(ndc_column_sums(out_fptr(partial), out_fptr(sums), partial.size(0), partial.size(1), stream), "ndc_column_sums");
    return sums;
}

// gz = gy * act'(z + bias), and the bias gradient from the values before they are rounded to gz's
// type (summing what is stored instead put a bf16 rounding into every term)
void act_backward(const Tensor &gy, const Tensor &z, const Tensor &bias, const Tensor &gz, int act, Tensor *gb, void *stream)
{
    const int64_t B = gy.size(0), C = gy.size(1), n = gy.size(2);
    Tensor partial;
    if (gb) partial = empty_f32({B, C, ndc_bias_act_parts(B * C, n)}, gy);
    check(ndc_bias_act_backward(ptr(gy), ptr(z), fptr(bias), out_ptr(gz), out_fptr(partial), B, C, n, act, dtype_tag(gy), stream),
          "ndc_bias_act_backward");
    if (gb) *gb = partial.sum(at::IntArrayRef{0, 2});
}

// ndc_weight_grad on tensors within its reach
Tensor weight_grad_within(const Tensor &a, const Tensor &c, Tensor *sums, void *stream)
{
    const int64_t B = a.size(0), n = a.size(2), rows = a.size(1), cols = c.size(1);
    Tensor gw = empty_f32({rows, cols}, a);
    if (sums) *sums = empty_f32({rows}, a);
    const int64_t bytes = (int64_t)ndc_weight_grad_workspace_bytes(B, rows, cols, n, dtype_tag(a));
    Tensor ws = bytes ? at::empty({bytes}, a.options().dtype(at::kByte)) : Tensor();
    check(ndc_weight_grad(ptr(a), ptr(c), out_fptr(gw), sums ? out_fptr(*sums) : nullptr, B, rows, cols, n, dtype_tag(a), out_ptr(ws),
                          bytes, stream), "ndc_weight_grad");
    return gw;
}

// Weight gradient sum_b gz[b] x[b]^T, (cout, cin) -- or (cin, cout) for a weight stored
// transposed --, and the bias gradient, the sums of gz, from the same pass.  The kernel's lane offsets
// reach 2^24 voxels; longer rows go through it slice by slice, copied (the slices of a row lie apart).
Tensor weight_grad(const Tensor &gz, const Tensor &x, const Matrix &w, at::IntArrayRef shape, at::ScalarType dtype, Tensor *gb,
                   void *stream)
{
    const Tensor &a = w.transposed ? x : gz, &c = w.transposed ? gz : x;
    const int64_t n = a.size(2), most = int64_t(1) << 24;
    Tensor gw, *sums = gb && !w.transposed ? gb : nullptr;
    if (n <= most) {
        gw = weight_grad_within(a, c, sums, stream);
    } else {
        const int64_t slices = (n + most - 1) / most, step = ((n + slices - 1) / slices + 127) / 128 * 128;
        for (int64_t lo = 0; lo < n; lo += step) {
            const int64_t len = std::min(step, n - lo);
            Tensor part;
            const Tensor g = weight_grad_within(a.narrow(2, lo, len).contiguous(), c.narrow(2, lo, len).contiguous(),
                                                sums ? &part : nullptr, stream);
            gw = lo ? gw.add_(g) : g;
            if (sums) *sums = lo ? sums->add_(part) : part;
        }
    }
    if (gb && !sums) *gb = channel_sums(gz, stream);
    return gw.to(dtype).view(shape);
}

// ---------------------------------------------------------------------------- the update

struct UpdateConfig {
    int64_t groups, m, sc;
    double eps;
    bool relu_input, save_ratio;
};

ndc_geom geom_for(const Tensor &x, const Tensor &h, const UpdateConfig &c, int path)
{
    ndc_geom g;
    const int rank = (int)x.dim() - 2;
    TORCH_CHECK_VALUE(rank >= 1 && rank <= 3 && h.dim() - 2 == rank, "unsupported spatial rank ", rank, " / kernel rank ",
                      h.dim() - 2);
    g.batch = (int32_t)x.size(0);
    g.groups = (int32_t)c.groups;
    g.m = (int32_t)c.m;
    g.sc = (int32_t)c.sc;
    for (int a = 0; a < 3; ++a) {
        const int d = a - (3 - rank);
        g.size[a] = d < 0 ? 1 : (int32_t)x.size(2 + d);
        g.kernel[a] = d < 0 ? 1 : (int32_t)h.size(2 + d);
    }
    g.dtype = dtype_tag(x);
    g.relu_input = c.relu_input ? 1 : 0;
    g.path = path;
    g.eps = (float)c.eps;
    return g;
}

void check_update(const Tensor &x, const Tensor &z, const Tensor &h, const Tensor &bias, const UpdateConfig &c)
{
    TORCH_CHECK_VALUE(x.dim() >= 3 && x.dim() <= 5, "expected a (B, C, *S) tensor with 1-3 spatial dims, got ", x.sizes());
    TORCH_CHECK_VALUE(x.size(1) == c.groups * c.m, "x has ", x.size(1), " channels, expected groups*m = ", c.groups * c.m);
    bool same = z.dim() == x.dim() && z.size(0) == x.size(0) && z.size(1) == c.groups * c.sc;
    for (int64_t d = 2; same && d < x.dim(); ++d) same = z.size(d) == x.size(d);
    TORCH_CHECK_VALUE(same, "z has shape ", z.sizes(), ", expected the extents of x ", x.sizes(), " with ", c.groups * c.sc,
                      " channels");
    TORCH_CHECK_VALUE(h.dim() == x.dim() && h.size(0) * h.size(1) == c.groups * c.m * c.sc, "filter of shape ", h.sizes(),
                      " does not match groups=", c.groups, ", m=", c.m, ", sc=", c.sc);
    TORCH_CHECK_TYPE(x.scalar_type() == z.scalar_type(), "x (", x.scalar_type(), ") and z (", z.scalar_type(),
                     ") must share a dtype");
    TORCH_CHECK_TYPE(h.scalar_type() == at::kFloat && (!bias.defined() || bias.scalar_type() == at::kFloat),
                     "filter and bias must be float32");
    for (const Tensor *t : {&x, &z, &h, &bias})
        TORCH_CHECK_VALUE(!t->defined() || (t->device() == x.device() && t->is_contiguous()),
                          "all tensors must be contiguous and on one device");
    TORCH_CHECK_VALUE(!bias.defined() || bias.numel() == c.groups * c.sc, "bias has ", bias.numel(), " entries, expected ",
                      c.groups * c.sc);
}

// a 256-byte aligned slice of a fresh buffer
Tensor scratch(size_t bytes, const Tensor &like)
{
    Tensor buf = at::empty({(int64_t)bytes + 256}, like.options().dtype(at::kByte));
    const int64_t off = (256 - (int64_t)((uintptr_t)buf.const_data_ptr() & 255)) & 255;
    return buf.narrow(0, off, (int64_t)bytes);
}

// max(h0, 0), and where no table is given the one the kernels of this geometry read
Tensor rectify_filter(const ndc_geom &g, const Tensor &h0, Tensor &taps, void *stream)
{
    const size_t bytes = taps.defined() ? 0 : ndc_taps_bytes(&g);
    Tensor h = at::empty_like(h0);
    if (bytes) taps = scratch(bytes, h0);
    check(ndc_rectify_filter(&g, fptr(h0), out_fptr(h), bytes ? out_ptr(taps) : nullptr, bytes, stream), "ndc_rectify_filter");
    return h;
}

// the filter table the kernels of this geometry read instead of h, or undefined
Tensor prepare_taps(const ndc_geom &g, const Tensor &h, void *stream)
{
    const size_t bytes = ndc_taps_bytes(&g);
    if (!bytes) return Tensor();
    Tensor taps = scratch(bytes, h);
    check(ndc_prepare_taps(&g, fptr(h), out_ptr(taps), bytes, stream), "ndc_prepare_taps");
    return taps;
}

void check_taps(const Tensor &taps, const Tensor &x, const ndc_geom &g)
{
    if (!taps.defined()) return;
    check_device(taps, x, "the filter table");
    TORCH_CHECK_VALUE(taps.is_contiguous() && taps.nbytes() >= ndc_taps_bytes(&g), "the filter table is another geometry's");
}

struct UpdateForward {
    Tensor x, z, t1, h, s_over_den, ratio, taps;   // what the backward reads (h: contiguous)
    int path;
    bool x_last, z_last;                           // x / z came in channels-last
};

// Forward of an update.  `grad`: a backward will follow.  `rectify`: h is the filter before its rectifier.
Tensor update_forward(Tensor x, Tensor z, const Tensor &h, const Tensor &bias, Tensor taps, const UpdateConfig &c, bool grad,
                      UpdateForward &f, void *stream, bool rectify = false)
{
    // channels-last tensors come in through the library's tiled transposition, and the results
    // go back out the same way, in the layout of the tensor they belong to
    f.x_last = channels_last(x);
    f.z_last = channels_last(z);
    x = channel_first(x, stream);
    z = channel_first(z, stream);
    Tensor hc = h.contiguous();
    check_update(x, z, hc, bias, c);
    // The kernel family is read once, here, and named in both calls of this node: backward runs
    // on an autograd thread, possibly after the process default has changed.
    ndc_geom g = geom_for(x, hc, c, NDC_PATH_AUTO);
    const bool fused = ndc_fused_supported(&g) != 0;
    if (fused) g.path = ndc_matrix_kernels(-1) ? NDC_PATH_FUSED_MATRIX : NDC_PATH_FUSED_VECTOR;
    f.path = g.path;
    // (kept only where the backward kernels of this geometry read them)
    const bool keep = grad && c.save_ratio && ndc_backward_uses_saved(&g);
    check_taps(taps, x, g);
    // packed once here, used by the forward kernel and again by the backward's
    if (rectify) hc = rectify_filter(g, hc, taps, stream);
    else if (!taps.defined()) taps = prepare_taps(g, hc, stream);
    Tensor out = at::empty_like(z);
    if (grad || !fused) f.t1 = at::empty_like(x);
    if (keep) {
        f.s_over_den = at::empty_like(z);
        f.ratio = at::empty_like(z);
    }
    if (taps.defined()) {
        check(ndc_forward_taps(&g, ptr(x), ptr(z), fptr(hc), ptr(taps), fptr(bias), out_ptr(out), out_ptr(f.t1),
                               out_ptr(f.s_over_den), out_ptr(f.ratio), stream), "ndc_forward_taps");
    } else {
        const size_t bytes = ndc_forward_workspace_bytes(&g);
        Tensor ws = bytes ? scratch(bytes, x) : Tensor();
        check(ndc_forward(&g, ptr(x), ptr(z), fptr(hc), fptr(bias), out_ptr(out), out_ptr(f.t1), out_ptr(f.s_over_den),
                          out_ptr(f.ratio), out_ptr(ws), bytes, stream), "ndc_forward");
    }
    f.x = x;
    f.z = z;
    f.h = hc;
    f.taps = taps;
    return f.z_last ? to_channels_last(out, stream) : out;
}

void refuse_double_backward(bool recording)
{
    // The gradients come from kernels autograd cannot see through, so a second differentiation
    // would silently drop terms: refuse it, as the reference does.
    TORCH_CHECK(!recording, "double backward through the fused Deconv update is not supported; construct the layer with a "
                            "convolution keyword argument (e.g. stride=1) to force the general path, which is plain PyTorch "
                            "and doubly differentiable");
}

struct UpdateGrads {
    Tensor gx, gz, gh, gb;
};

UpdateGrads update_backward(const UpdateForward &f, const Tensor &bias, Tensor gout, const UpdateConfig &c, bool need_x,
                            bool need_z, bool need_h, bool need_b, void *stream, bool rectify = false)
{
    const Tensor &x = f.x, &z = f.z;
    check_update(x, z, f.h, bias, c);
    const Tensor t1 = check_saved(f.t1, x), s_over_den = check_saved(f.s_over_den, z), ratio = check_saved(f.ratio, z);
    if (gout.scalar_type() != z.scalar_type()) gout = gout.to(z.scalar_type());
    gout = channel_first(gout, stream);
    TORCH_CHECK_VALUE(gout.sizes() == z.sizes(), "the gradient has shape ", gout.sizes(), ", expected ", z.sizes());
    need_b = need_b && bias.defined();
    const ndc_geom g = geom_for(x, f.h, c, f.path);
    UpdateGrads r;
    if (need_x) r.gx = at::empty_like(x);
    if (need_z) r.gz = at::empty_like(z);
    if (need_h) r.gh = at::empty_like(f.h);
    if (need_b) r.gb = empty_f32({c.groups * c.sc}, x);
    const size_t bytes = ndc_backward_workspace_bytes(&g, need_x, need_z, need_h, need_b);
    Tensor ws = scratch(bytes ? bytes : 1, x);
    check_taps(f.taps, x, g);
    if (rectify)
        check(ndc_backward_rectified(&g, ptr(x), ptr(z), ptr(t1), ptr(s_over_den), ptr(ratio), fptr(f.h), ptr(f.taps),
                                     fptr(bias), ptr(gout), out_ptr(r.gx), out_ptr(r.gz), out_fptr(r.gh), out_fptr(r.gb),
                                     out_ptr(ws), bytes, stream), "ndc_backward_rectified");
    else if (f.taps.defined())
        check(ndc_backward_taps(&g, ptr(x), ptr(z), ptr(t1), ptr(s_over_den), ptr(ratio), fptr(f.h), ptr(f.taps),
                                fptr(bias), ptr(gout), out_ptr(r.gx), out_ptr(r.gz), out_fptr(r.gh), out_fptr(r.gb),
                                out_ptr(ws), bytes, stream), "ndc_backward_taps");
    else
        check(ndc_backward(&g, ptr(x), ptr(z), ptr(t1), ptr(s_over_den), ptr(ratio), fptr(f.h), fptr(bias), ptr(gout),
                           out_ptr(r.gx), out_ptr(r.gz), out_fptr(r.gh), out_fptr(r.gb), out_ptr(ws), bytes, stream),
              "ndc_backward");
    return r;
}

void save_config(AutogradContext *ctx, const UpdateConfig &c, const UpdateForward &f)
{
    ctx->saved_data["cfg"] = std::vector<int64_t>{c.groups, c.m, c.sc, c.relu_input, f.path, f.x_last, f.z_last};
    ctx->saved_data["eps"] = c.eps;
}

void load_config(AutogradContext *ctx, UpdateConfig &c, UpdateForward &f)
{
    const auto v = ctx->saved_data["cfg"].toIntVector();
    c = UpdateConfig{v[0], v[1], v[2], ctx->saved_data["eps"].toDouble(), v[3] != 0, false};
    f.path = (int)v[4];
    f.x_last = v[5] != 0;
    f.z_last = v[6] != 0;
}

// out = relu?(z + b) * (A(x) + eps) / (A(K(relu?(z + b))) + eps)
struct Update : public torch::autograd::Function<Update> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &z, const Tensor &h, const OptTensor &bias,
                          const OptTensor &taps, const UpdateConfig &c)
    {
        Scope scope(x);
        UpdateForward f;
        const Tensor b = bias ? *bias : Tensor();
        Tensor out = update_forward(x, z, h, b, taps ? *taps : Tensor(), c, true, f, scope.stream);
        save_config(ctx, c, f);
        ctx->save_for_backward({f.x, f.z, f.t1, f.h, b, f.s_over_den, f.ratio, f.taps});
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        refuse_double_backward(at::GradMode::is_enabled());
        UpdateConfig c;
        UpdateForward f;
        load_config(ctx, c, f);
        const auto v = ctx->get_saved_variables();
        f.x = v[0], f.z = v[1], f.t1 = v[2], f.h = v[3], f.s_over_den = v[5], f.ratio = v[6], f.taps = v[7];
        Scope scope(f.x);
        Needs n;
        n.arg(true), n.arg(true), n.arg(true), n.arg(v[4].defined());
        const auto need = n.ask(ctx);
        UpdateGrads r = update_backward(f, v[4], gouts[0], c, need[0], need[1], need[2], need[3], scope.stream);
        if (f.x_last && r.gx.defined()) r.gx = to_channels_last(r.gx, scope.stream);
        if (f.z_last && r.gz.defined()) r.gz = to_channels_last(r.gz, scope.stream);
        return {r.gx, r.gz, r.gh, r.gb, Tensor(), Tensor()};
    }
};

Tensor update(const Tensor &x, const Tensor &z, const Tensor &h, const OptTensor &bias, int64_t groups, int64_t m, int64_t sc,
              double eps, bool relu_input, const OptTensor &taps, bool save_ratio)
{
    no_tangents(x, z, h, bias);
    const UpdateConfig c{groups, m, sc, eps, relu_input, save_ratio};
    if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(z) || wants_grad(h) || wants_grad(bias)))
        return Update::apply(x, z, h, bias, taps, c);
    Scope scope(x);
    UpdateForward f;
    return update_forward(x, z, h, bias ? *bias : Tensor(), taps ? *taps : Tensor(), c, false, f, scope.stream);
}

// Whether a bare float32 product that widens -- a layer's projection, an upsampling -- is the tiled GEMM's: those
// below half a GFLOP, and up to one from at most 128 channels.  A call of the library takes the host 10-18 us longer,
// and on the GPU the tiled GEMM is ahead or within 2 us there (us, library / tiled: 32 -> 128 channels over 4096 voxels
// 5.3 / 4.5, over 36 608 12.9 / 9.1; 64 -> 256 over 9152 10.3 / 8.8; 48 -> 192 over 36 608 37.6 / 15.0; 128 -> 256 over
// 143 29 / 4.0, over 4096 6.9 / 8.0; 256 -> 1024 over 572 9.0 / 10.0; behind from there on: 512 -> 1024 over 572, 0.6
// GFLOP, 11.3 / 16.4, 512 -> 2048 17 / 24).  It is nearer to 64 bits too (32 to 512 channels 0.7e-7 to 1.6e-7 of the
// result's norm, the library 1.0e-7 to 4.1e-7).  Past a GFLOP the library's product stays also where it is behind: its
// bits decide which source units are on, and what else forms the product of a large network -- a check of its on/off
// patterns by torch.bmm -- sees the same units.  Samples count with the columns of 64 voxels they fill.
// One 208 x 176 image through the 2-D network, forward: 1.24 -> 0.95 ms; a layer of 32 channels of 64^2 with its
// backward 0.180 -> 0.150.
bool wide_is_tiled(int64_t B, int64_t cin, int64_t cout, int64_t n)
{
    // (no parts: nothing to do, or more than the tiled GEMM takes)
    if (cin >= cout || !ndc_gemm_parts(B, cin, cout, n, NDC_F32)) return false;
    const double columns = (double)B * (double)((n + 63) / 64 * 64), flops = 2.0 * (double)cin * (double)cout * columns;
    return flops < 0.5e9 || (cin <= 128 && flops < 1e9);
}

// The layer's first update together with the 1x1 projection that makes its source
// (deconv.py:157-165 with layers/linear.py:53-58 of the reference): z = W x per sample, then the
// update of (x, z) with the projection's bias and the ReLU applied where the kernels load z.  One
// node because x feeds both: as two nodes their input gradients are two tensors that autograd
// adds in a pass of its own; here the projection's input-gradient GEMM accumulates onto the
// update's gx.  With `rectify` the node takes the filter parameter itself and rectifies it (the
// filter's relu and its backward are then no nodes of their own).
struct Projected : public torch::autograd::Function<Projected> {
    static Tensor run(const Tensor &x_, const Tensor &weight, const Tensor &h, const Tensor &bias, const Tensor &taps,
                      const UpdateConfig &c, bool grad, bool rectify, UpdateForward &f, void *stream)
    {
        const Matrix w(weight, false);
        // (the GEMMs and the update read rows of voxels: any other layout is turned first)
        const Tensor x = channel_first(x_, stream);
        auto size = x.sizes().vec();
        const Tensor flat = x.flatten(2);
        const bool library = x.scalar_type() == at::kFloat && !wide_is_tiled(flat.size(0), w.cin(), w.cout(), flat.size(2));
        Tensor z = project(w, flat, library, stream);
        size[1] = w.cout();
        Tensor out = update_forward(x, z.view(size), rectify ? h.detach() : h, bias, taps, c, grad, f, stream, rectify);
        f.x_last = channels_last(x_);
        return out;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight, const Tensor &h, const OptTensor &bias,
                          const OptTensor &taps, const UpdateConfig &c, bool rectified_input, bool rectify)
    {
        Scope scope(x);
        UpdateForward f;
        const Tensor b = bias ? *bias : Tensor();
        Tensor out = run(x, weight, h, b, taps ? *taps : Tensor(), c, true, rectify, f, scope.stream);
        save_config(ctx, c, f);
        ctx->saved_data["flags"] = std::vector<int64_t>{rectified_input, rectify};
        ctx->save_for_backward({f.x, f.z, f.t1, f.h, b, f.s_over_den, f.ratio, f.taps, weight});
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        refuse_double_backward(at::GradMode::is_enabled());
        UpdateConfig c;
        UpdateForward f;
        load_config(ctx, c, f);
        const auto flags = ctx->saved_data["flags"].toIntVector();
        const auto v = ctx->get_saved_variables();
        f.x = v[0], f.z = v[1], f.t1 = v[2], f.h = v[3], f.s_over_den = v[5], f.ratio = v[6], f.taps = v[7];
        Scope scope(f.x);
        Needs n;
        n.arg(true), n.arg(true), n.arg(true), n.arg(v[4].defined());
        const auto need = n.ask(ctx);
        UpdateGrads r =
            update_backward(f, v[4], gouts[0], c, need[0], need[0] || need[1], need[2], need[3], scope.stream, flags[1] != 0);
        const Tensor x = f.x.flatten(2);
        const Matrix w = saved_weight(v[8], false, f.z.size(1), x);
        TORCH_CHECK_VALUE(w.cin() == x.size(1), "a saved weight came back as ", v[8].sizes());
        Tensor gw, gx;
        if (need[1]) gw = weight_grad(r.gz.flatten(2), x, w, v[8].sizes(), v[8].scalar_type(), nullptr, scope.stream);
        if (need[0]) {
            gx = project_back(w, r.gz.flatten(2), r.gx.flatten(2), flags[0] ? x : Tensor(), scope.stream).view(f.x.sizes());
            if (f.x_last) gx = to_channels_last(gx, scope.stream);
        }
        return {gx, gw, r.gh, r.gb, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

Tensor projected_update(const Tensor &x, const Tensor &weight, const Tensor &h, const OptTensor &bias, int64_t groups,
                        int64_t m, int64_t sc, double eps, const OptTensor &taps, bool rectified_input, bool rectify,
                        bool save_ratio)
{
    no_tangents(x, weight, h, bias);
    TORCH_CHECK_VALUE(x.dim() >= 3 && x.dim() <= 5, "expected a (B, C, *S) tensor with 1-3 spatial dims, got ", x.sizes());
    check_projection(x, x.size(1), weight, false, bias, OptTensor());
    check_device(h, x, "the filter");
    const UpdateConfig c{groups, m, sc, eps, true, save_ratio};
    if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(weight) || wants_grad(h) || wants_grad(bias)))
        return Projected::apply(x, weight, h, bias, taps, c, rectified_input, rectify);
    Scope scope(x);
    UpdateForward f;
    return Projected::run(x, weight, h, bias ? *bias : Tensor(), taps ? *taps : Tensor(), c, false, rectify, f, scope.stream);
}

// ---------------------------------------------------------------------------- projection with its tail

// Whether a bare float32 product that narrows (a stage's adapter, a downsampling; nobody's but its node's) is
// the tiled GEMM's.  Up to some 250 voxels a sample the library has one workgroup for each, whose time grows with
// them, and is ahead where many samples fill the chip with those while the tiled GEMM's 64-voxel columns are part
// empty.  us, library / tiled: 512 -> 256 channels over 256 voxels 119 / 6, over 16 x 256 119 / 18, over 128 x 16
// 22 / 30, over 64 x 4 13 / 17; 384 -> 192 over 241 82 / 5.3; 256 -> 128 over 64 x 16 9.5 / 6.0, over 256 x 16 9.4 / 18;
// 768 -> 384 over 16 x 128 14 / 23, 1024 -> 512 over 16 6.4 / 8.3.  Beyond that the library is ahead in larger products:
// 512 -> 256 over 500 7.1 / 6.2, over 1024 7.3 / 8.2, over 2048 9.1 / 14.7; 384 -> 192 over 1840 7.8 / 9.8, over 2714
// 8.2 / 13.5; 1024 -> 512 over 500 9.9 / 13.4.  2 us more on the GPU (0.3 GFLOP) are less than the 10 us that a call of
// the library takes the host longer: the 2-D network's forward on one 208 x 176 image, whose four adapters are 0.15
// GFLOP each, takes 1.34 ms with theirs by the library and 1.23 tiled.
bool narrow_is_tiled(int64_t B, int64_t cin, int64_t cout, int64_t n)
{
    if (cin <= cout) return false;
    const double weights = 2.0 * (double)cin * (double)cout, least = 0.3e9;
    if (n > 256) return weights * (double)B * (double)n < least;
    const int64_t columns = B * ((n + 63) / 64 * 64);
    if (columns > 4200 + 145 * n) return false;
    return weights * (double)columns < least || (cin <= 512 && (n >= 16 || weights * (double)columns < 1e9));
}

// y[b] = act(W x[b] + bias) + residual[b] on channel-first (B, C, n) tensors.  keep: the
// activation's gradient will want the product (gelu, or relu under a residual sum)
struct Linear : public torch::autograd::Function<Linear> {
    static Tensor run(const Tensor &x, const Matrix &w, const Tensor &bias, int64_t act, const Tensor &res, bool keep, Tensor &z,
                      void *stream)
    {
        const int64_t B = x.size(0), n = x.size(2), cout = w.cout();
        const bool tail = bias.defined() || act != NDC_ACT_NONE || res.defined();
        // An activation's tile form reads W as rows.  A bare float32 product that widens could be a layer's
        // projection taken apart: the same product, bit for bit, as in Projected.
        const bool bare = !tail && x.scalar_type() == at::kFloat;
        const bool library = (w.transposed && act != NDC_ACT_NONE) ||
                             (bare && !narrow_is_tiled(B, w.cin(), cout, n) && !wide_is_tiled(B, w.cin(), cout, n));
        const Gemm by = library ? kLibrary : choose_gemm(x, cout, act != NDC_ACT_NONE || keep, tail);
        Tensor y = empty({B, cout, n}, x);
        if (keep) z = empty({B, cout, n}, x);
        if (by == kStream) {
            // product, bias, activation and residual in one kernel that reads x once and writes
            // the result (and z where it is kept) once
            Tensor frag = pack(w, false, x, stream);
            check(ndc_pointwise_gemm(ptr(x), ptr(frag), fptr(bias), ptr(res), out_ptr(y), out_ptr(z), B, w.cin(), cout, n,
                                     (int)act, NDC_BF16, stream), "ndc_pointwise_gemm");
        } else if (by == kTiled) {
            tiled(w, false, x, bias, res, Tensor(), y, z, (int)act, stream);
        } else {
            Tensor &product = keep ? z : y;
            at::bmm_out(product, batched(w.dense(x.scalar_type(), false), B), x);
            if (tail)
                check(ndc_bias_act(ptr(product), fptr(bias), ptr(res), out_ptr(y), B, cout, n, (int)act, dtype_tag(x), stream),
                      "ndc_bias_act");
        }
        return y;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight, const OptTensor &bias, int64_t act,
                          const OptTensor &residual, bool premasked, bool transposed)
    {
        Scope scope(x);
        const Matrix w(weight, transposed);
        const Tensor b = f32_vector(bias), res = residual ? *residual : Tensor();
        // relu alone needs only the sign of its output
        const bool keep = act == NDC_ACT_GELU || (act == NDC_ACT_RELU && res.defined());
        Tensor z;
        Tensor y = run(x, w, b, act, res, keep, z, scope.stream);
        ctx->save_for_backward({x, weight, keep ? z : act == NDC_ACT_RELU ? y : Tensor(), keep ? b : Tensor()});
        // (premasked: every gradient that arrives is already zero where the result is)
        ctx->saved_data["cfg"] = std::vector<int64_t>{
            act, bias.has_value() && bias->defined(), res.defined(), premasked && act == NDC_ACT_RELU && !res.defined(), transposed,
            bias.has_value() && bias->defined() ? (int64_t)bias->scalar_type() : 0};
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto cfg = ctx->saved_data["cfg"].toIntVector();
        const int act = (int)cfg[0];
        const auto v = ctx->get_saved_variables();
        const Tensor gy = gouts[0].contiguous();
        Scope scope(gy);
        const Matrix w = saved_weight(v[1], cfg[4] != 0, gy.size(1), gy);
        const Tensor x = check_saved(v[0], gy, {gy.size(0), w.cin(), gy.size(2)}, gy.scalar_type());
        const Tensor kept = check_saved(v[2], gy), bias = check_saved(v[3], gy, {w.cout()}, at::kFloat);
        Needs n;
        n.arg(true), n.arg(true), n.arg(cfg[1]), n.arg(cfg[2]);
        const auto need = n.ask(ctx);
        Tensor gz = gy, gx, gw, gb;
        if (act != NDC_ACT_NONE && !cfg[3]) {
            gz = at::empty_like(gy);
            // (a rectifier's gradient, and float32, are stored as they are: their sums come with the weight's)
            const bool rounded = act == NDC_ACT_GELU && gy.scalar_type() == at::kBFloat16;
            act_backward(gy, kept, bias, gz, act, need[2] && rounded ? &gb : nullptr, scope.stream);
        }
        Tensor *sums = need[2] && !gb.defined() ? &gb : nullptr;
        if (need[0]) gx = project_back(w, gz, Tensor(), Tensor(), scope.stream);
        if (need[1]) gw = weight_grad(gz, x, w, v[1].sizes(), v[1].scalar_type(), sums, scope.stream);
        else if (sums) gb = channel_sums(gz, scope.stream);
        if (gb.defined()) gb = gb.to((at::ScalarType)cfg[5]);
        return once({gx, gw, gb, Tensor(), need[3] ? gy : Tensor(), Tensor(), Tensor()}, recording, gouts);
    }
};

Tensor linear(const Tensor &x, const Tensor &weight, const OptTensor &bias, int64_t act, const OptTensor &residual,
              bool premasked, bool transposed)
{
    no_tangents(x, weight, bias, residual);
    TORCH_CHECK_VALUE(x.dim() == 3, "expected a (B, C, n) tensor, got ", x.sizes());
    check_projection(x, x.size(1), weight, transposed, bias, residual);
    const Tensor xc = x.contiguous();
    OptTensor res = residual;
    if (res && res->defined()) {
        if (res->scalar_type() != xc.scalar_type()) res = res->to(xc.scalar_type());
        res = res->contiguous();
    }
    if (at::GradMode::is_enabled() && (wants_grad(xc) || wants_grad(weight) || wants_grad(bias) || wants_grad(res)))
        return Linear::apply(xc, weight, bias, act, res, premasked, transposed);
    Scope scope(xc);
    Tensor z;
    return Linear::run(xc, Matrix(weight, transposed), f32_vector(bias), act, res ? *res : Tensor(), false, z, scope.stream);
}

// Whether an MLP runs with its hidden tensor on chip (ndc_mlp_forward / _backward) where those kernels
// apply: with 64 channels from 32 768 voxels on (their kernels take 24 + 30 us there, the projections' 30 +
// 55; over 16 384 voxels 23 against 20 forward), with 32 from 4096 (7.5 + 15 against 8.1 + 23).
int64_t mlp_least_voxels(int64_t c) { return c == 32 ? 4096 : 32768; }

bool mlp_on_chip(const Tensor &x, const Matrix &w1, const Matrix &w2)
{
    const int64_t c = x.size(1), n = x.size(2);
    auto type = [](const Tensor &t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; };
    return x.scalar_type() == at::kBFloat16 && w1.cout() == 4 * c && w2.cout() == c && type(w1.m) && w1.m.scalar_type() == w2.m.scalar_type() &&
           x.size(0) * n >= mlp_least_voxels(c) && ndc_mlp_supported(c, n, NDC_BF16) && ((uintptr_t)ptr(x) & 3) == 0;
}

// the tensor at an address the kernels' 16-byte accesses take
Tensor aligned(const Tensor &t) { return ((uintptr_t)ptr(t) & 15) ? t.clone() : t; }

// W2 gelu(W1 x + b1) + b2 + residual on contiguous (B, C, n) tensors (layers/mlp.py:40-63 with the
// block's sum, deconver.py:60-64).  Where mlp_on_chip says so the hidden tensor never leaves the chip: one
// kernel forward, and one backward that forms it again from x.  Elsewhere the GELU and the kept
// pre-activation leave the first product, bias and residual ride on the second, and in backward the
// input gradient of the second comes out already multiplied by the GELU's derivative where one of the
// library's own GEMMs makes it.
struct Mlp : public torch::autograd::Function<Mlp> {
    static Tensor run(const Tensor &x, const Matrix &w1, const Tensor &b1, const Matrix &w2, const Tensor &b2, const Tensor &res,
                      bool keep, bool on_chip, Tensor &z, Tensor &a, void *stream)
    {
        if (on_chip && (!res.defined() || ((uintptr_t)ptr(res) & 3) == 0)) {
            Tensor y = empty(x.sizes(), x);
            check(ndc_mlp_forward(ptr(x), nullptr, ptr(w1.m), ptr(w2.m), dtype_tag(w1.m), fptr(b1), fptr(b2), ptr(res), out_ptr(y), x.size(0),
                                  x.size(1), x.size(2), NDC_BF16, stream), "ndc_mlp_forward");
            return y;
        }
        Tensor unused;
        a = Linear::run(x, w1, b1, NDC_ACT_GELU, Tensor(), keep, z, stream);
        return Linear::run(a, w2, b2, NDC_ACT_NONE, res, false, unused, stream);
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w1, const OptTensor &b1, const Tensor &w2,
                          const OptTensor &b2, const OptTensor &residual)
    {
        Scope scope(x);
        Tensor z, a;
        const Tensor b1f = f32_vector(b1);
        const Matrix m1(w1, false), m2(w2, false);
        // (the backward forms the hidden tensor again, which pays where all gradients may be wanted)
        const bool on_chip = wants_grad(x) && wants_grad(w1) && wants_grad(w2) && mlp_on_chip(x, m1, m2);
        Tensor y = run(x, m1, b1f, m2, f32_vector(b2), residual ? *residual : Tensor(), true, on_chip, z, a, scope.stream);
        ctx->save_for_backward({x, z, a, w1, w2, b1f});   // (z, a undefined: the hidden tensor stayed on chip)
        ctx->saved_data["cfg"] = std::vector<int64_t>{b1.has_value(), b2.has_value(), residual.has_value(),
                                                      b1 ? (int64_t)b1->scalar_type() : 0, b2 ? (int64_t)b2->scalar_type() : 0};
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto cfg = ctx->saved_data["cfg"].toIntVector();
        const auto v = ctx->get_saved_variables();
        const Tensor gy = gouts[0].contiguous();
        Scope scope(gy);
        const Matrix w2 = saved_weight(v[4], false, gy.size(1), gy), w1 = saved_weight(v[3], false, w2.cin(), gy);
        const int64_t B = gy.size(0), nv = gy.size(2), hidden = w1.cout();
        const Tensor x = check_saved(v[0], gy, {B, w1.cin(), nv}, gy.scalar_type());
        const Tensor b1 = check_saved(v[5], gy, {hidden}, at::kFloat);
        Needs n;
        n.arg(true), n.arg(true), n.arg(cfg[0]), n.arg(true), n.arg(cfg[1]), n.arg(cfg[2]);
        const auto need = n.ask(ctx);
        Tensor gx, gw1, gb1, gw2, gb2;
        if (!v[1].defined()) {
            // (the kernels know the widths by x's channels alone)
            TORCH_CHECK_VALUE(hidden == 4 * x.size(1) && w2.cout() == x.size(1), "saved weights came back as ", v[3].sizes(), " and ",
                              v[4].sizes(), " for an MLP of ", x.size(1), " channels with four times as many hidden ones");
            const Tensor xa = aligned(x), ga = aligned(gy);
            const bool half = w1.m.scalar_type() == at::kBFloat16 && w2.m.scalar_type() == at::kBFloat16;
            const Tensor m1 = half ? w1.m : w1.m.to(at::kFloat), m2 = half ? w2.m : w2.m.to(at::kFloat);
            if (need[0]) gx = empty(x.sizes(), x);
            if (need[1]) gw1 = empty_f32(m1.sizes(), x);
            if (need[3]) gw2 = empty_f32(m2.sizes(), x);
            if (need[2]) gb1 = empty_f32({hidden}, x);
            if (need[4]) gb2 = empty_f32({w2.cout()}, x);
            const size_t bytes = ndc_mlp_workspace_bytes(B, x.size(1), nv);
            Tensor ws = scratch(bytes, x);
            check(ndc_mlp_backward(ptr(xa), ptr(ga), ptr(m1), ptr(m2), dtype_tag(m1), fptr(b1), out_ptr(gx), out_fptr(gw1), out_fptr(gb1),
                                   out_fptr(gw2), out_fptr(gb2), B, x.size(1), nv, NDC_BF16, out_ptr(ws), bytes, scope.stream),
                  "ndc_mlp_backward");
            if (gb1.defined()) gb1 = gb1.to((at::ScalarType)cfg[3]);
            if (gb2.defined()) gb2 = gb2.to((at::ScalarType)cfg[4]);
            if (gw1.defined()) gw1 = gw1.to(v[3].scalar_type()).view(v[3].sizes());
            if (gw2.defined()) gw2 = gw2.to(v[4].scalar_type()).view(v[4].sizes());
            return once({gx, gw1, gb1, gw2, gb2, need[5] ? gy : Tensor()}, recording, gouts);
        }
        const Tensor z = check_saved(v[1], gy, {B, hidden, nv}, gy.scalar_type()), a = check_saved(v[2], z);
        if (need[3]) gw2 = weight_grad(gy, a, w2, v[4].sizes(), v[4].scalar_type(), need[4] ? &gb2 : nullptr, scope.stream);
        else if (need[4]) gb2 = channel_sums(gy, scope.stream);
        if (need[0] || need[1] || need[2]) {
            // bf16: the first bias's gradient is summed in the kernels that make gz, before they round
            // it (what they store carries a rounding in every term); float32: with the weight's
            Tensor gz = at::empty_like(z);
            const bool rounded = need[2] && gy.scalar_type() == at::kBFloat16;
            const Gemm by = choose_gemm(gy, hidden, true, true);
            Tensor partial;
            if (by == kStream) {
                Tensor frag = pack(w2, true, gy, scope.stream);
                if (rounded) partial = empty_f32({ndc_pointwise_gemm_parts(), hidden}, gy);
                check(ndc_pointwise_gemm_actgrad(ptr(gy), ptr(frag), fptr(b1), ptr(z), out_ptr(gz), out_fptr(partial), B, w2.cout(),
                                                 hidden, nv, NDC_ACT_GELU, NDC_BF16, scope.stream), "ndc_pointwise_gemm_actgrad");
            } else if (by == kTiled) {
                const Tensor m = w2.m.to(at::kFloat);
                if (rounded) partial = empty_f32({ndc_gemm_parts(B, w2.cout(), hidden, nv, dtype_tag(gy)), hidden}, gy);
                check(ndc_gemm_gelu_grad(ptr(gy), fptr(m), fptr(b1), ptr(z), out_ptr(gz), out_fptr(partial), B, w2.cout(), hidden, nv,
                                         dtype_tag(gy), scope.stream), "ndc_gemm_gelu_grad");
            } else {
                Tensor ga = project_back(w2, gy, Tensor(), Tensor(), scope.stream);
                act_backward(ga, z, b1, gz, NDC_ACT_GELU, rounded ? &gb1 : nullptr, scope.stream);
            }
            if (partial.defined()) gb1 = column_sums(partial, scope.stream);
            Tensor *sums = need[2] && !gb1.defined() ? &gb1 : nullptr;
            if (need[1]) gw1 = weight_grad(gz, x, w1, v[3].sizes(), v[3].scalar_type(), sums, scope.stream);
            else if (sums) gb1 = channel_sums(gz, scope.stream);
            if (need[0]) gx = project_back(w1, gz, Tensor(), Tensor(), scope.stream);
        }
        if (gb1.defined()) gb1 = gb1.to((at::ScalarType)cfg[3]);
        if (gb2.defined()) gb2 = gb2.to((at::ScalarType)cfg[4]);
        return once({gx, gw1, gb1, gw2, gb2, need[5] ? gy : Tensor()}, recording, gouts);
    }
};

Tensor mlp(const Tensor &x, const Tensor &w1, const OptTensor &b1, const Tensor &w2, const OptTensor &b2,
           const OptTensor &residual)
{
    no_tangents(x, w1, b1, w2, b2, residual);
    TORCH_CHECK_VALUE(x.dim() == 3, "expected a (B, C, n) tensor, got ", x.sizes());
    const int64_t hidden = check_projection(x, x.size(1), w1, false, b1, OptTensor());
    check_projection(x, hidden, w2, false, b2, residual);
    const Tensor xc = x.contiguous();
    OptTensor res = residual;
    if (res && res->defined()) {
        if (res->scalar_type() != xc.scalar_type()) res = res->to(xc.scalar_type());
        res = res->contiguous();
    }
    if (at::GradMode::is_enabled() && (wants_grad(xc) || wants_grad(w1) || wants_grad(b1) || wants_grad(w2) || wants_grad(b2) ||
                                       wants_grad(res)))
        return Mlp::apply(xc, w1, b1, w2, b2, res);
    Scope scope(xc);
    Tensor z, a;
    const Matrix m1(w1, false), m2(w2, false);
    return Mlp::run(xc, m1, f32_vector(b1), m2, f32_vector(b2), res ? *res : Tensor(), false, mlp_on_chip(xc, m1, m2), z, a,
                    scope.stream);
}

// ---------------------------------------------------------------------------- norms

Tensor row_workspace(int64_t rows, int64_t n, const Tensor &like)
{
    return empty_f32({std::max<int64_t>((int64_t)ndc_rownorm_workspace_bytes(rows, n) / 4, 2)}, like);
}

Tensor row_norm_forward(const Tensor &x, double eps, Tensor &stats, void *stream)
{
    const int64_t rows = x.size(0) * x.size(1), n = voxels(x);
    Tensor y = at::empty_like(x);
    stats = empty_f32({rows, 2}, x);
    Tensor ws = row_workspace(rows, n, x);
    check(ndc_rownorm_forward(ptr(x), out_ptr(y), out_fptr(stats), rows, n, dtype_tag(x), (float)eps, out_ptr(ws), ws.numel() * 4,
                              stream), "ndc_rownorm_forward");
    return y;
}

Tensor row_norm_backward(const Tensor &gy, const Tensor &saved_y, const Tensor &saved_stats, const Tensor &addend, void *stream)
{
    const Tensor y = check_saved(saved_y, gy), stats = check_saved(saved_stats, gy, {gy.size(0) * gy.size(1), 2}, at::kFloat);
    const int64_t rows = stats.size(0), n = voxels(y);
    Tensor gx = at::empty_like(y), ws = row_workspace(rows, n, y);
    check(ndc_rownorm_backward(ptr(gy), ptr(y), fptr(stats), ptr(addend), out_ptr(gx), rows, n, dtype_tag(y), out_ptr(ws),
                               ws.numel() * 4, stream), "ndc_rownorm_backward");
    return gx;
}

struct RowNorm : public torch::autograd::Function<RowNorm> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, double eps)
    {
        Scope scope(x);
        Tensor stats, y = row_norm_forward(x.contiguous(), eps, stats, scope.stream);
        ctx->save_for_backward({y, stats});
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto v = ctx->get_saved_variables();
        Scope scope(gouts[0]);
        return once({row_norm_backward(gouts[0].contiguous(), v[0], v[1], Tensor(), scope.stream), Tensor()}, recording, gouts);
    }
};

// (norm(x), x) for a pre-norm residual block x + f(norm(x)): in backward the gradient that
// arrives for the second output is summed into the norm's own input gradient by the kernel that
// writes it, instead of by a separate addition
struct RowNormSkip : public torch::autograd::Function<RowNormSkip> {
    static variable_list forward(AutogradContext *ctx, const Tensor &x, double eps)
    {
        // (outside the scope: below it a view is an alias without a base and with a version of its own,
        // whose changes in place autograd would not see)
        const Tensor skip = x.view_as(x);
        Scope scope(x);
        Tensor stats, y = row_norm_forward(x.contiguous(), eps, stats, scope.stream);
        ctx->save_for_backward({y, stats});
        ctx->set_materialize_grads(false);   // an unused output's gradient arrives undefined
        return {y, skip};
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto v = ctx->get_saved_variables();
        if (!gouts[0].defined()) return {gouts[1], Tensor()};
        Scope scope(gouts[0]);
        Tensor skip = gouts[1];
        if (skip.defined()) skip = skip.to(gouts[0].scalar_type()).contiguous();
        return once({row_norm_backward(gouts[0].contiguous(), v[0], v[1], skip, scope.stream), Tensor()}, recording, gouts);
    }
};

Tensor row_norm(const Tensor &x, double eps)
{
    no_tangents(x);
    if (at::GradMode::is_enabled() && wants_grad(x)) return RowNorm::apply(x, eps);
    Scope scope(x);
    Tensor stats;
    return row_norm_forward(x.contiguous(), eps, stats, scope.stream);
}

std::pair<Tensor, Tensor> row_norm_skip(const Tensor &x, double eps)
{
    no_tangents(x);
    if (!at::GradMode::is_enabled() || !wants_grad(x)) return {row_norm(x, eps), x};
    auto r = RowNormSkip::apply(x, eps);
    return {r[0], r[1]};
}

// nn.LayerNorm over the channel axis of a channel-first (B, C, n) tensor: lanes along the
// voxels, a loop over the channels, nothing transposed
struct ChannelNorm : public torch::autograd::Function<ChannelNorm> {
    static Tensor run(const Tensor &x, const Tensor &w, const Tensor &b, double eps, Tensor &stats, void *stream)
    {
        const int64_t B = x.size(0), C = x.size(1), n = x.size(2);
        Tensor y = at::empty_like(x);
        stats = empty_f32({B, 2, n}, x);
        check(ndc_chnorm_forward(ptr(x), fptr(w), fptr(b), out_ptr(y), out_fptr(stats), B, C, n, dtype_tag(x), (float)eps, stream),
              "ndc_chnorm_forward");
        return y;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const OptTensor &weight, const OptTensor &bias, double eps)
    {
        Scope scope(x_);
        const Tensor x = x_.contiguous(), w = f32_vector(weight), b = f32_vector(bias);
        Tensor stats, y = run(x, w, b, eps, stats, scope.stream);
        ctx->save_for_backward({x, stats, w});
        ctx->saved_data["cfg"] = std::vector<int64_t>{weight.has_value(), bias.has_value(),
                                                      weight ? (int64_t)weight->scalar_type() : 0,
                                                      bias ? (int64_t)bias->scalar_type() : 0};
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto cfg = ctx->saved_data["cfg"].toIntVector();
        const auto v = ctx->get_saved_variables();
        const Tensor gy = gouts[0].contiguous();
        Scope scope(gy);
        const int64_t B = gy.size(0), C = gy.size(1), n = gy.size(2);
        const Tensor x = check_saved(v[0], gy), stats = check_saved(v[1], gy, {B, 2, n}, at::kFloat);
        const Tensor weight = check_saved(v[2], gy, {C}, at::kFloat);
        Needs nd;
        nd.arg(true), nd.arg(cfg[0]), nd.arg(cfg[1]);
        const auto need = nd.ask(ctx);
        Tensor gx = at::empty_like(x), partial, gw, gb;
        const bool affine = need[1] || need[2];
        if (affine) partial = empty_f32({ndc_chnorm_parts(B, n, dtype_tag(x)), C, 2}, x);
        check(ndc_chnorm_backward(ptr(gy), ptr(x), fptr(stats), fptr(weight), out_ptr(gx), out_fptr(partial), B, C, n, dtype_tag(x),
                                  scope.stream), "ndc_chnorm_backward");
        if (affine) {
            // (the library's own sum, two launches of 4 us: torch's takes 10 and clears a semaphore ahead of it, 4 more)
            // Its columns end at 2^22; more than half as many channels take torch's.
            const Tensor sums = 2 * C > (1 << 22) ? partial.sum(0)
                                                  : column_sums(partial.view({partial.size(0), 2 * C}), scope.stream).view({C, 2});
            if (need[1]) gw = sums.select(1, 0).to((at::ScalarType)cfg[2]).contiguous();
            if (need[2]) gb = sums.select(1, 1).to((at::ScalarType)cfg[3]).contiguous();
        }
        return once({need[0] ? gx : Tensor(), gw, gb, Tensor()}, recording, gouts);
    }
};

Tensor channel_norm(const Tensor &x, const OptTensor &weight, const OptTensor &bias, double eps)
{
    no_tangents(x, weight, bias);
    TORCH_CHECK_VALUE(x.dim() == 3, "expected a (B, C, n) tensor, got ", x.sizes());
    check_vector(weight, x, x.size(1), "the weight");
    check_vector(bias, x, x.size(1), "the bias");
    if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(weight) || wants_grad(bias)))
        return ChannelNorm::apply(x, weight, bias, eps);
    Scope scope(x);
    Tensor stats;
    return ChannelNorm::run(x.contiguous(), f32_vector(weight), f32_vector(bias), eps, stats, scope.stream);
}

// ---------------------------------------------------------------------------- regrouping

// 2 x 2 (x 2) windows of the grid <-> 2^nd channels per window; each direction's gradient is the
// other direction.  On the way back to the grid a per-channel bias can be added in the same pass.
Tensor regroup_run(const Tensor &x, bool to_channels, const Tensor &bias, void *stream)
{
    const int64_t B = x.size(0), nd = x.dim() - 2, win = int64_t(1) << nd;
    auto size = x.sizes().vec();
    size[1] = to_channels ? x.size(1) * win : x.size(1) / win;
    for (int64_t d = 0; d < nd; ++d) size[2 + d] = to_channels ? x.size(2 + d) / 2 : x.size(2 + d) * 2;
    Tensor out = empty(size, x);
    const auto fine = to_channels ? x.sizes() : out.sizes();
    const int64_t C = fine[1], D = nd == 3 ? fine[2] : 1;
    check(ndc_regroup(ptr(x), out_ptr(out), fptr(bias), B * C, C, D, fine[nd], fine[nd + 1], nd == 3, dtype_tag(x), to_channels,
                      stream), "ndc_regroup");
    return out;
}

struct Regroup : public torch::autograd::Function<Regroup> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, bool to_channels, const OptTensor &bias)
    {
        Scope scope(x);
        ctx->saved_data["cfg"] = std::vector<int64_t>{to_channels, bias.has_value() && bias->defined(),
                                                      bias && bias->defined() ? (int64_t)bias->scalar_type() : 0};
        return regroup_run(x, to_channels, f32_vector(bias), scope.stream);
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const bool recording = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const auto cfg = ctx->saved_data["cfg"].toIntVector();
        const Tensor g = gouts[0].contiguous();
        Scope scope(g);
        Needs n;
        n.arg(true), n.arg(cfg[1]);
        const auto need = n.ask(ctx);
        Tensor gb;
        if (!cfg[0] && need[1]) gb = channel_sums(g.flatten(2), scope.stream).to((at::ScalarType)cfg[2]);
        return once({regroup_run(g, !cfg[0], Tensor(), scope.stream), Tensor(), gb}, recording, gouts);
    }
};

Tensor regroup(const Tensor &x, bool to_channels, const OptTensor &bias)
{
    no_tangents(x, bias);
    TORCH_CHECK_VALUE((x.dim() == 4 || x.dim() == 5) && x.is_contiguous(),
                      "expected a contiguous (B, C, *S) tensor with 2-3 spatial dims, got ", x.sizes());
    const int64_t window = int64_t(1) << (x.dim() - 2);
    TORCH_CHECK_VALUE(to_channels || x.size(1) % window == 0, "expected a multiple of ", window, " channels, got ", x.sizes());
    check_vector(bias, x, x.size(1) / window, "the bias");
    if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(bias))) return Regroup::apply(x, to_channels, bias);
    Scope scope(x);
    return regroup_run(x, to_channels, f32_vector(bias), scope.stream);
}

// ---------------------------------------------------------------------------- training loss

// Cross-entropy plus Dice loss (ndc_loss.h) of float32 (B, C, *S) logits and targets of their shape.
struct DiceBce : public torch::autograd::Function<DiceBce> {
    static Tensor run(const Tensor &l, const Tensor &y, Tensor &coef, void *stream)
    {
        const int64_t rows = l.size(0) * l.size(1), n = l.numel() / rows;
        Tensor loss = empty_f32({}, l);
        coef = empty_f32({rows, 2}, l);
        const size_t bytes = ndc_dice_bce_workspace_bytes(rows, n);
        Tensor ws = empty_f32({(int64_t)(bytes / 4)}, l);
        check(ndc_dice_bce_forward(fptr(l), fptr(y), out_fptr(loss), out_fptr(coef), rows, n, out_ptr(ws), bytes, stream),
              "ndc_dice_bce_forward");
        return loss;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &l, const Tensor &y)
    {
        Scope scope(l);
        Tensor coef, loss = run(l.contiguous(), y.contiguous(), coef, scope.stream);
        ctx->save_for_backward({l, y, coef});
        return loss;
    }
    // (under create_graph the gradient is made of tensor operations, which can be differentiated again)
    static Tensor formula(const Tensor &l, const Tensor &y_, const Tensor &g)
    {
        const int64_t rows = l.size(0) * l.size(1), n = l.numel() / rows;
        const Tensor p = l.reshape({rows, n}).sigmoid(), y = y_.reshape({rows, n});
        const Tensor num = 2 * (p * y).sum(1, true) + 1, den = p.sum(1, true) + y.sum(1, true) + 1;
        const Tensor dp = (num / (den * den) - 2 * y / den) / (double)rows;
        return (g * ((p - y) / ((double)rows * (double)n) + p * (1 - p) * dp)).view(l.sizes());
    }
    static variable_list backward(AutogradContext *ctx, variable_list gouts)
    {
        const auto v = ctx->get_saved_variables();
        const Tensor &g = gouts[0];
        check_device(v[0], g, "a saved tensor");
        const c10::DeviceGuard device(g.device());
        if (at::GradMode::is_enabled() && (wants_grad(g) || wants_grad(v[0]))) return {formula(v[0], v[1], g), Tensor()};
        Scope scope(g);
        TORCH_CHECK_VALUE(v[0].dim() >= 3 && v[0].numel() > 0, "a saved tensor came back as ", v[0].sizes());
        const int64_t rows = v[0].size(0) * v[0].size(1), n = v[0].numel() / rows;
        const Tensor l = check_saved(v[0], g, v[0].sizes(), at::kFloat), y = check_saved(v[1], g, l.sizes(), at::kFloat);
        const Tensor coef = check_saved(v[2], g, {rows, 2}, at::kFloat), gl = at::empty_like(l);
        check(ndc_dice_bce_backward(fptr(l), fptr(y), fptr(coef), fptr(g.contiguous()), out_fptr(gl), rows, n, scope.stream),
              "ndc_dice_bce_backward");
        return {gl, Tensor()};
    }
};

// None for tensors that the kernels do not take; the caller has the loss in tensor operations.
OptTensor dice_bce(const Tensor &l, const Tensor &y)
{
    const auto plain = [](const Tensor &t) {
        return t.is_cuda() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided && !t._fw_grad(0).defined() &&
               !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize}));
    };
    if (!plain(l) || !plain(y) || l.device() != y.device() || l.dim() < 3 || l.sizes() != y.sizes() || l.numel() == 0 ||
        wants_grad(y) || ndc_dice_bce_workspace_bytes(l.size(0) * l.size(1), voxels(l)) == 0)
        return std::nullopt;
    if (at::GradMode::is_enabled() && wants_grad(l)) return DiceBce::apply(l, y);
    Scope scope(l);
    Tensor coef;
    return DiceBce::run(l.contiguous(), y.contiguous(), coef, scope.stream);
}

// ---------------------------------------------------------------------------- optimiser

// One AdamW step in place, or false, with nothing done, where a tensor is not what the kernel takes
// (dense float32 of one device, the gradient and the moments laid out as the parameter).
bool adamw(const std::vector<Tensor> &params, const std::vector<Tensor> &grads, const std::vector<Tensor> &m,
           const std::vector<Tensor> &v, const std::vector<Tensor> &steps, double lr, double beta1, double beta2, double eps,
           double weight_decay)
{
    const size_t count = params.size();
    if (!count) return true;
    if (grads.size() != count || m.size() != count || v.size() != count || steps.size() != count) return false;
    const auto device = params[0].device();
    const auto plain = [&](const Tensor &t) {
        return t.defined() && t.device() == device && t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == at::kFloat &&
               !t.is_conj() && !t.is_neg() && !t.key_set().has(c10::DispatchKey::Python);
    };
    std::vector<ndc_adamw_tensor> list(count);
    for (size_t i = 0; i < count; ++i) {
        for (const Tensor *t : {&params[i], &grads[i], &m[i], &v[i]})
            if (!plain(*t) || !t->is_contiguous() || t->sizes() != params[i].sizes()) return false;
        if (!plain(steps[i]) || steps[i].numel() != 1) return false;
    }
    Scope scope(params[0]);
    for (size_t i = 0; i < count; ++i) {
        list[i] = {out_fptr(params[i]), fptr(grads[i]), out_fptr(m[i]), out_fptr(v[i]), out_fptr(steps[i]), params[i].numel()};
        for (const Tensor *t : {&params[i], &m[i], &v[i], &steps[i]}) t->unsafeGetTensorImpl()->bump_version();
    }
    check(ndc_adamw(list.data(), (int64_t)count, lr, beta1, beta2, eps, weight_decay, scope.stream), "ndc_adamw");
    return true;
}

// ---------------------------------------------------------------------------- columns

// Column matrix of a contiguous (B, C, *S) tensor for odd kernel extents k: (B, C * taps, voxels).
// Not differentiable: the caller takes it for inputs that need no gradient.
Tensor columns(const Tensor &x, const std::vector<int64_t> &k)
{
    no_tangents(x);
    const int64_t nd = x.dim() - 2;
    TORCH_CHECK_VALUE(nd >= 1 && nd <= 3 && (int64_t)k.size() == nd && x.is_contiguous(),
                      "expected a contiguous (B, C, *S) tensor and one odd extent per spatial dim, got ", x.sizes());
    Scope scope(x);
    int64_t size[3] = {1, 1, 1}, ext[3] = {1, 1, 1}, taps = 1, n = 1;
    for (int64_t d = 0; d < nd; ++d) {
        size[3 - nd + d] = x.size(2 + d), ext[3 - nd + d] = k[d];
        taps *= k[d], n *= x.size(2 + d);
    }
    Tensor out = empty({x.size(0), x.size(1) * taps, n}, x);
    check(ndc_columns(ptr(x), out_ptr(out), x.size(0) * x.size(1), size[0], size[1], size[2], (int)ext[0], (int)ext[1],
                      (int)ext[2], dtype_tag(x), scope.stream), "ndc_columns");
    return out;
}

OptTensor taps_for(const Tensor &x, const Tensor &h, int64_t groups, int64_t m, int64_t sc)
{
    TORCH_CHECK_TYPE(h.scalar_type() == at::kFloat, "the filter must be float32");
    TORCH_CHECK_VALUE(h.numel() > 0 && h.dim() >= 3 && h.size(0) * h.size(1) == groups * m * sc && h.is_contiguous(),
                      "filter of shape ", h.sizes(), " does not match groups=", groups, ", m=", m, ", sc=", sc);
    check_device(h, x, "the filter");
    Scope scope(x);
    const ndc_geom g = geom_for(x, h, UpdateConfig{groups, m, sc, 0.0, true, false}, NDC_PATH_AUTO);
    Tensor taps = prepare_taps(g, h, scope.stream);
    return taps.defined() ? OptTensor(taps) : OptTensor();
}

// ---------------------------------------------------------------------------- a block in one call

// x + mixer(norm(x)), then y + mlp(norm(y)) (deconver.py:49-65 of the reference) out of the nodes above, in the
// order and with the operands of the modules' own calls; None where a layer's geometry is not the kernels'.
// What a call saves is the modules between the nodes, some 70 us of Python a block where a small block's
// kernels take as long: the 2-D network's forward on one 208 x 176 image 1.78 -> 1.18 ms, a training step on a
// 32^3 volume, whose pace is the host's, from 4.4-5.2 ms to 2.7-3.9.
OptTensor block(const Tensor &x_, bool half, double eps1, double eps2, const Tensor &w_in, const OptTensor &b_in, const Tensor &h0,
                const Tensor &w_source, const OptTensor &b_source, int64_t groups, int64_t m, int64_t sc, double eps, bool save_ratio,
                const Tensor &w_out, const OptTensor &b_out, const Tensor &w1, const OptTensor &b1, const Tensor &w2,
                const OptTensor &b2)
{
    const at::ScalarType dtype = half ? at::kBFloat16 : at::kFloat;
    Tensor x = x_;
    if (x.dim() < 3 || x.dim() > 5 || h0.dim() != x.dim() || w_in.size(0) != groups * m) return std::nullopt;
    ndc_geom g = geom_for(x, h0, UpdateConfig{groups, m, sc, 0.0, true, false}, NDC_PATH_AUTO);
    g.dtype = half ? NDC_BF16 : NDC_F32;
    if (ndc_check_geometry(&g) != 0) return std::nullopt;
    const auto cast = [&](const Tensor &t) { return t.scalar_type() == dtype ? t : t.to(dtype); };
    const auto grid = [&](const Tensor &t, int64_t channels) {
        auto size = x_.sizes().vec();
        size[1] = channels;
        return t.view(size);
    };
    const auto normed = [&](double e, Tensor &residual) {
        if (!wants_grad(residual)) return row_norm(residual, e);
        auto r = row_norm_skip(residual, e);
        residual = r.second;
        return r.first;
    };
    // Calls without a backward behind them normalise where the projections load, with the same bits: rows of
    // more than 192 KB, which no workgroup holds, whose norm would be a pass to reduce and another to write
    // what the projection reads again.  The 3-D network's forward on one 96 x 128 x 112 volume 6.49 -> 6.19 ms.
    bool plain = half && x.scalar_type() == at::kBFloat16 && voxels(x) > 12 * 8192 && x.is_contiguous() && ((uintptr_t)ptr(x) & 3) == 0;
    for (const Tensor *t : {&x_, &w_in, &h0, &w_source, &w_out, &w1, &w2}) plain = plain && !(at::GradMode::is_enabled() && wants_grad(*t));
    for (const OptTensor *t : {&b_in, &b_source, &b_out, &b1, &b2}) plain = plain && !(at::GradMode::is_enabled() && wants_grad(*t));
    const int64_t B = x.size(0), C = x.size(1), n = voxels(x);
    const Matrix m_in(w_in, false), m1(w1, false), m2(w2, false);
    const auto streams = [&](int64_t cin, const Matrix &w, int act) {
        return w.cin() == cin && ndc_pointwise_gemm_normed_supported(cin, w.cout(), n, act) && B * n >= 2048 * 64;
    };
    const auto statistics = [&](const Tensor &t, double e, void *stream) {
        Tensor stats = empty_f32({B * C, 2}, t), ws = row_workspace(B * C, n, t);
        check(ndc_rownorm_stats(ptr(t), out_fptr(stats), B * C, n, NDC_BF16, (float)e, out_ptr(ws), ws.numel() * 4, stream),
              "ndc_rownorm_stats");
        return stats;
    };
    const auto normed_projection = [&](const Tensor &t, const Tensor &stats, const Matrix &w, const OptTensor &bias, int act, void *stream) {
        check_vector(bias, t, w.cout(), "the bias");
        Tensor out = empty({B, w.cout(), n}, t), frag = pack(w, false, t, stream);
        const Tensor b = f32_vector(bias);
        check(ndc_pointwise_gemm_normed(ptr(t), fptr(stats), ptr(frag), fptr(b), out_ptr(out), B, w.cin(), w.cout(), n, act, NDC_BF16,
                                        stream), "ndc_pointwise_gemm_normed");
        return out;
    };
    Tensor y;
    const bool fold1 = plain && streams(C, m_in, NDC_ACT_RELU);
    if (fold1) {
        no_tangents(x, w_in, b_in);
        check_device(w_in, x, "the weight");
        Scope scope(x);
        y = normed_projection(x, statistics(x, eps1, scope.stream), m_in, b_in, NDC_ACT_RELU, scope.stream);
    } else {
        y = normed(eps1, x);
    }
    // (the rectifier's backward rides on the layer's input gradient where that is one streaming GEMM)
    const bool premasked = half && x.size(1) == groups * m && ndc_pointwise_gemm_supported(groups * sc, groups * m, voxels(x), NDC_BF16);
    if (!fold1) y = linear(cast(y.flatten(2)), w_in, b_in, NDC_ACT_RELU, std::nullopt, premasked, false);
    y = grid(y, w_in.size(0));
    OptTensor bias = b_source;
    if (bias && bias->scalar_type() != at::kFloat) bias = bias->to(at::kFloat);
    y = projected_update(y.contiguous(), w_source, h0, bias, groups, m, sc, eps, std::nullopt, premasked, true, save_ratio);
    x = grid(linear(cast(y.flatten(2)), w_out, b_out, NDC_ACT_NONE, x.flatten(2), false, false), w_out.size(0));
    if (plain && x.is_contiguous() && x.size(1) == C && m1.cin() == C && m2.cin() == m1.cout() && m2.cout() == C) {
        const Tensor flat = x.flatten(2);
        const bool on_chip = mlp_on_chip(flat, m1, m2);
        if (on_chip || streams(C, m1, NDC_ACT_GELU)) {
            no_tangents(x, w1, b1, w2, b2);
            check_device(w1, x, "the weight"), check_device(w2, x, "the weight");
            check_vector(b1, x, m1.cout(), "the bias"), check_vector(b2, x, C, "the bias");
            Scope scope(x);
            const Tensor stats = statistics(x, eps2, scope.stream);
            if (!on_chip)
                return grid(linear(normed_projection(flat, stats, m1, b1, NDC_ACT_GELU, scope.stream), w2, b2, NDC_ACT_NONE, flat, false, false), C);
            const Tensor bf1 = f32_vector(b1), bf2 = f32_vector(b2);
            y = at::empty_like(x);
            check(ndc_mlp_forward(ptr(x), fptr(stats), ptr(m1.m), ptr(m2.m), dtype_tag(m1.m), fptr(bf1), fptr(bf2), ptr(x), out_ptr(y), B,
                                  C, n, NDC_BF16, scope.stream), "ndc_mlp_forward");
            return y;
        }
    }
    y = normed(eps2, x);
    return grid(mlp(cast(y.flatten(2)), w1, b1, w2, b2, x.flatten(2)), w2.size(0));
}

// the name Python shows for a node (type(y.grad_fn))
template <class F> void name_node(const char *name)
{
    static PyTypeObject type{};
    torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
    torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<F>), &type);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    name_node<Update>("DeconvUpdateBackward");
    name_node<Projected>("ProjectedUpdateBackward");
    name_node<Linear>("_PointwiseLinearBackward");
    name_node<Mlp>("_FusedMLPBackward");
    name_node<RowNorm>("_RowNormBackward");
    name_node<RowNormSkip>("_RowNormSkipBackward");
    name_node<ChannelNorm>("_ChannelNormBackward");
    name_node<Regroup>("_RegroupBackward");
    name_node<DiceBce>("_DiceBceBackward");
    m.def("update", &update);
    m.def("projected_update", &projected_update);
    m.def("prepare_taps", &taps_for);
    m.def("linear", &linear);
    m.def("mlp", &mlp);
    m.def("row_norm", &row_norm);
    m.def("row_norm_skip", &row_norm_skip);
    m.def("channel_norm", &channel_norm);
    m.def("regroup", &regroup);
    m.def("columns", &columns);
    m.def("dice_bce", &dice_bce);
    m.def("adamw", &adamw);
    m.def("block", &block);
}
