// Direct kernels: the general path, for any rank / grouping / kernel extent (geometries the fused
// LDS-tiled kernels do not cover) and the on-GPU cross-check of the fused kernels.
//
// Tap conventions (deconver/deconvolution/kernels.py:32-39 of the reference):
//   K(u)[o,p] = sum_{i,tau} u[i, p + tau - pad] * h[o,i,tau]
//   A(v)[i,p] = sum_{o,tau} v[o, p + pad - tau] * h[o,i,tau]
//
// A thread owns one position of one (sample, group) and a block of NB output channels; lanes run
// along the positions.  A value of a neighbour is loaded once and used for all NB channels, its
// weights are the same in every lane and come through the scalar unit or, where a launch has the
// wavefronts (Weights::staged), from a copy in LDS in the order they are used -- each channel's few
// adjacent weights are a short scalar load of their own, and the scalar cache, which two CUs share,
// was what large launches waited for --, and the window's address
// and bounds are formed once per tap row and serve every input channel.  One thread per output
// element, which this replaces, repeated each load, its 64-bit address and its bounds branch for
// every output channel.  The filter gradient holds MB x SB x KWB sums (filter channels x source
// channels x taps of a row) and walks the positions, so that each load feeds three products; one
// workgroup per single sum loaded two values a product and read the volume m*sc*taps times.
// What bounds these kernels now is the load path of the CU (a 4-byte load of a wavefront takes
// four clocks, as a multiply-add of its four SIMDs does) and, in small launches, the weights'
// latency; the volumes they serve fit the L2.
// Measured (4 groups of 4 filter and 8 source channels, 3x3x3, 2 x 24^3, float32): t1 94 -> 35 us,
// the forward's ratio 89 -> 25, gn and gd 65 -> 26, gx and gt1 145 -> 26, gh 419 -> 41, gz 151 -> 36,
// gb 41 -> 5; the layer, forward + backward, 1036 -> 236 us.  Filters of 3 x 3 and 5 x 5 taps take their
// convolutions from boxes in LDS since (ndc_direct_tile.h); 1-D ones, those of unequal extents, of 7 taps
// and volumes past what its boxes cover (some 130^3 or 300^2) are done here.
#pragma once

#include "../../include/deconver_ndc.h"
#include "ndc_common.h"

namespace ndc {
namespace direct {

// OFF: the type of byte offsets inside one channel's volume (uint32_t below 2^32 bytes of float)
template <typename T, typename OFF> NDC_HD float load_at(const T *base, OFF idx)
{
    return Elem<T>::load((const T *)((const char *)base + (OFF)(idx * (OFF)sizeof(T))));
}

template <typename OFF> struct Pos {
    int d, h, w;
    OFF off;
};

template <typename OFF> NDC_HD Pos<OFF> position(const KGeom &q, OFF p)
{
    Pos<OFF> r;
    r.off = p;
    r.w = (int)(p % (OFF)q.W);
    p /= (OFF)q.W;
    r.h = (int)(p % (OFF)q.H);
    r.d = (int)(p / (OFF)q.H);
    return r;
}

// The row of taps (td, th) and its taps tw0 .. tw0 + KWB around a position, as K (SIGN = 1) or A
// (SIGN = -1) reads it: offsets inside a channel, and whether they lie in the volume.  Taps
// outside are given the position itself (in bounds) and are not counted.
template <int SIGN, int KWB, typename OFF> struct Window {
    OFF at[KWB];
    bool in[KWB];
    NDC_HD Window(const KGeom &q, const Pos<OFF> &p, int td, int th, int tw0)
    {
        const int dd = p.d + SIGN * (td - q.pD), hh = p.h + SIGN * (th - q.pH);
        const bool row_in = (unsigned)dd < (unsigned)q.D && (unsigned)hh < (unsigned)q.H;
        const OFF row = ((OFF)(row_in ? dd : p.d) * (OFF)q.H + (OFF)(row_in ? hh : p.h)) * (OFF)q.W;
#pragma unroll
        for (int j = 0; j < KWB; ++j) {
            const int ww = p.w + SIGN * (tw0 + j - q.pW);
            in[j] = row_in && (unsigned)ww < (unsigned)q.W;
            at[j] = row + (OFF)(in[j] ? ww : p.w);
        }
    }
    template <typename T> NDC_HD void load(const T *channel, float (&v)[KWB]) const
    {
#pragma unroll
        for (int j = 0; j < KWB; ++j) {
            const float t = load_at<T, OFF>(channel, at[j]);
            v[j] = in[j] ? t : 0.f;
        }
    }
};

// The weights that output channels c0 .. c0 + NB of a group take, in the order accumulate() takes them:
// [taps by KWB][input channel][output channel][KWB].  A workgroup puts them into LDS where they fit.
static const int kStagedWeights = 4096;
template <bool ADJ, int NB, int KWB> struct Weights {
    // Whether a launch of so many wavefronts takes n weights from LDS (16 KB at most).  us, scalar unit -> LDS,
    // float32: forwards of 2 groups of 4 -> 16 channels on 64^3 273 -> 161, 8 of 1 -> 8 on 48^3 150 -> 98, 8 of
    // 1 -> 4 with 7x7 taps on 8 x 128^2 276 -> 216.  With few wavefronts the copy and the LDS's latency show:
    // A of 4 -> 8 channels on 2 x 24^3 (3456 wavefronts of 4 outputs) 25 -> 34, K 35 -> 31; both of 16 -> 16 on
    // 24^3 (1728 wavefronts) 73 -> 121.
    static bool staged(int n, long long waves)
    {
        return n <= kStagedWeights && (ADJ ? waves * NB >= 24 * 1024 : waves >= 3 * 1024);
    }
    static NDC_HD int count(const KGeom &q) { return (ADJ ? q.m : q.sc) * NB * q.KT; }
    // the NB x KWB weights of every `step`-th pair (taps, input channel)
    static NDC_HD void stage(const KGeom &q, const float *hf, int g, int c0, float *to, int first, int step)
    {
        const int cin = ADJ ? q.m : q.sc, cout = ADJ ? q.sc : q.m, pairs = q.KT / KWB * cin;
        const float *hg = hf + (long long)g * q.m * q.sc * q.KT;
        for (int r = first; r < pairs; r += step) {
            const int t = r / cin, ci = r - t * cin;
            float v[NB * KWB];
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const int k = c0 + c < cout ? c0 + c : cout - 1;
#pragma unroll
                for (int j = 0; j < KWB; ++j) v[c * KWB + j] = hg[((ADJ ? ci : k) * q.sc + (ADJ ? k : ci)) * q.KT + t * KWB + j];
            }
#pragma unroll
            for (int i = 0; i < NB * KWB; ++i) to[r * NB * KWB + i] = v[i];
        }
    }
};

// acc[k][c] += the sums of K (ADJ = false, outputs: the m channels) or A (ADJ = true, outputs: the
// sc channels) at one position for output channels c0 .. c0 + NB of group g and NIN inputs at once.
// load(k, channel, window, v): the window of input k.  Channels past the last repeat the last.
// STAGED: staged holds the weights as Weights has them.
template <bool ADJ, int NB, int KWB, int NIN, bool STAGED, typename OFF, class Load>
NDC_HD void accumulate(const KGeom &q, const float *hf, const float *staged, int g, int c0, const Pos<OFF> &p,
                       float (&acc)[NIN][NB], Load load)
{
    const int cin = ADJ ? q.m : q.sc, cout = ADJ ? q.sc : q.m;
    if constexpr (STAGED) {
#pragma unroll
        for (int k = 0; k < NIN; ++k)
#pragma unroll
            for (int c = 0; c < NB; ++c) acc[k][c] = 0.f;
        const float *w = staged;
        for (int td = 0; td < q.kD; ++td)
            for (int th = 0; th < q.kH; ++th)
                for (int tw0 = 0; tw0 < q.kW; tw0 += KWB) {
                    const Window<ADJ ? -1 : 1, KWB, OFF> win(q, p, td, th, tw0);
#pragma unroll 2
                    for (int ci = 0; ci < cin; ++ci, w += NB * KWB) {
                        float v[NIN][KWB];
#pragma unroll
                        for (int k = 0; k < NIN; ++k) load(k, ci, win, v[k]);
#pragma unroll
                        for (int c = 0; c < NB; ++c)
#pragma unroll
                            for (int j = 0; j < KWB; ++j)
#pragma unroll
                                for (int k = 0; k < NIN; ++k) acc[k][c] += v[k][j] * w[c * KWB + j];
                    }
                }
        return;
    }
    const UniformF hg = as_uniform(hf + (long long)g * q.m * q.sc * q.KT);
    int chan[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        const int k = c0 + c < cout ? c0 + c : cout - 1;
        chan[c] = (ADJ ? k : k * q.sc) * q.KT;
    }
    const int step = (ADJ ? q.sc : 1) * q.KT;
#pragma unroll
    for (int k = 0; k < NIN; ++k)
#pragma unroll
        for (int c = 0; c < NB; ++c) acc[k][c] = 0.f;
    for (int td = 0; td < q.kD; ++td)
        for (int th = 0; th < q.kH; ++th)
            for (int tw0 = 0; tw0 < q.kW; tw0 += KWB) {
                const Window<ADJ ? -1 : 1, KWB, OFF> win(q, p, td, th, tw0);
                const int tap = (td * q.kH + th) * q.kW + tw0;
#pragma unroll 2
                for (int ci = 0; ci < cin; ++ci) {
                    float v[NIN][KWB];
#pragma unroll
                    for (int k = 0; k < NIN; ++k) load(k, ci, win, v[k]);
#pragma unroll
                    for (int c = 0; c < NB; ++c)
#pragma unroll
                        for (int j = 0; j < KWB; ++j) {
                            const float wv = hg[chan[c] + ci * step + tap + j];
#pragma unroll
                            for (int k = 0; k < NIN; ++k) acc[k][c] += v[k][j] * wv;
                        }
                }
            }
}

// rectified, biased source value
NDC_HD float source_of(float v, float b, int relu)
{
    v += b;
    return relu && v < 0.f ? 0.f : v;   // a NaN stays a NaN, as in torch.relu
}

// which (sample, group, first output channel) a unit of `blocks` channel blocks is
struct Unit {
    int b, g, c0;
    NDC_HD Unit(int u, int G, int blocks, int nb)
    {
        c0 = u % blocks * nb;
        u /= blocks;
        g = u % G;
        b = u / G;
    }
};

// ---------------------------------------------------------------- grouped convolution
// ADJ = false: out (B,G*m,S) = K(in (B,G*sc,S));  ADJ = true: out (B,G*sc,S) = A(in (B,G*m,S)).
// When `rectify` is set the input is read as relu?(in + bias) (zero outside the volume).
template <typename TI, typename TO, bool ADJ, int NB, int KWB, typename OFF> struct GConv {
    KGeom q;
    const TI *in;
    const float *hf, *bias;
    int rectify;
    TO *out;
    int blocks;
    typedef direct::Weights<ADJ, NB, KWB> Weights;
    static constexpr bool kAdj = ADJ;
    static constexpr int kNin = 1, kNB = NB, kKWB = KWB;
    NDC_HD float value(int, const Unit &t, int ci, OFF off) const
    {
        const int cin = ADJ ? q.m : q.sc;
        const float v = load_at<TI, OFF>(in + (((long long)t.b * q.G + t.g) * cin + ci) * q.SP, off);
        return rectify ? source_of(v, bias ? bias[t.g * cin + ci] : 0.f, q.relu) : v;
    }
    NDC_HD void finish(const Unit &t, long long pos, const float (&acc)[1][NB]) const
    {
        const int cout = ADJ ? q.sc : q.m;
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (t.c0 + c < cout) Elem<TO>::store(out + (((long long)t.b * q.G + t.g) * cout + t.c0 + c) * q.SP + pos, acc[0][c]);
    }
    NDC_HD int weights() const { return Weights::count(q); }
    NDC_HD void stage(int u, float *to, int first, int step) const
    {
        const Unit t(u, q.G, blocks, NB);
        Weights::stage(q, hf, t.g, t.c0, to, first, step);
    }
    template <bool STAGED> NDC_HD void run(int u, long long pos, const float *staged) const
    {
        const Unit t(u, q.G, blocks, NB);
        const int cin = ADJ ? q.m : q.sc;
        const Pos<OFF> p = position<OFF>(q, (OFF)pos);
        const long long bg = (long long)t.b * q.G + t.g;
        const TI *ig = in + bg * cin * q.SP;
        float acc[1][NB];
        accumulate<ADJ, NB, KWB, 1, STAGED, OFF>(q, hf, staged, t.g, t.c0, p, acc,
                                                 [&](int, int ci, const Window<ADJ ? -1 : 1, KWB, OFF> &win, float (&v)[KWB]) {
            win.template load<TI>(ig + ci * q.SP, v);
            if (!rectify) return;
            const float bv = bias ? bias[t.g * cin + ci] : 0.f;
#pragma unroll
            for (int j = 0; j < KWB; ++j) v[j] = win.in[j] ? source_of(v[j], bv, q.relu) : 0.f;
        });
        finish(t, pos, acc);
    }
};

// gt1 = K(gd) and gx = K(gn) side by side: the same weights
template <typename T, int NB, int KWB, typename OFF> struct GradPair {
    KGeom q;
    const float *gn, *gd, *hf;
    T *gx;
    float *gt1;
    int blocks;
    typedef direct::Weights<false, NB, KWB> Weights;
    static constexpr bool kAdj = false;
    static constexpr int kNin = 2, kNB = NB, kKWB = KWB;
    NDC_HD float value(int k, const Unit &t, int ci, OFF off) const
    {
        return load_at<float, OFF>((k ? gd : gn) + (((long long)t.b * q.G + t.g) * q.sc + ci) * q.SP, off);
    }
    NDC_HD void finish(const Unit &t, long long pos, const float (&acc)[2][NB]) const
    {
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (t.c0 + c < q.m) {
                const long long at = (((long long)t.b * q.G + t.g) * q.m + t.c0 + c) * q.SP + pos;
                Elem<T>::store(gx + at, acc[0][c]);
                gt1[at] = acc[1][c];
            }
    }
    NDC_HD int weights() const { return Weights::count(q); }
    NDC_HD void stage(int u, float *to, int first, int step) const
    {
        const Unit t(u, q.G, blocks, NB);
        Weights::stage(q, hf, t.g, t.c0, to, first, step);
    }
    template <bool STAGED> NDC_HD void run(int u, long long pos, const float *staged) const
    {
        const Unit t(u, q.G, blocks, NB);
        const Pos<OFF> p = position<OFF>(q, (OFF)pos);
        const long long bg = (long long)t.b * q.G + t.g, base = bg * q.sc * q.SP;
        float acc[2][NB];
        accumulate<false, NB, KWB, 2, STAGED, OFF>(q, hf, staged, t.g, t.c0, p, acc,
                                                   [&](int k, int ci, const Window<1, KWB, OFF> &win, float (&v)[KWB]) {
            win.template load<float>((k ? gd : gn) + base + ci * q.SP, v);
        });
        finish(t, pos, acc);
    }
};

// ---------------------------------------------------------------- the elementwise stages
// n = A(x)+eps, d = A(t1)+eps at a position and NB source channels, then
//   FWD    out = s n / d, and s/d, n/d where asked for
//   GRAD   gn = g s / d, gd = -gn n / d (float scratch)
//   SOURCE gz = [z+b>0] (g n / d + A(gt1))
enum { FWD, GRAD, SOURCE };

template <typename T, int STAGE, int NB, int KWB, typename OFF> struct Ratio {
    KGeom q;
    const T *x, *t1, *z, *gout;
    const float *gt1, *hf, *bias;
    T *out, *s_over_den, *ratio;    // FWD; SOURCE writes gz to `out`
    float *gn, *gd;                 // GRAD
    int blocks;
    typedef direct::Weights<true, NB, KWB> Weights;
    static constexpr bool kAdj = true;
    static constexpr int kNin = STAGE == SOURCE ? 3 : 2, kNB = NB, kKWB = KWB;
    NDC_HD float value(int k, const Unit &t, int ci, OFF off) const
    {
        const long long at = (((long long)t.b * q.G + t.g) * q.m + ci) * q.SP;
        return k == 2 ? load_at<float, OFF>(gt1 + at, off) : load_at<T, OFF>((k ? t1 : x) + at, off);
    }
    NDC_HD int weights() const { return Weights::count(q); }
    NDC_HD void stage(int u, float *to, int first, int step) const
    {
        const Unit t(u, q.G, blocks, NB);
        Weights::stage(q, hf, t.g, t.c0, to, first, step);
    }
    template <bool STAGED> NDC_HD void run(int u, long long pos, const float *staged) const
    {
        const Unit t(u, q.G, blocks, NB);
        const Pos<OFF> p = position<OFF>(q, (OFF)pos);
        const long long bg = (long long)t.b * q.G + t.g, base = bg * q.m * q.SP;
        float acc[kNin][NB];
        accumulate<true, NB, KWB, kNin, STAGED, OFF>(q, hf, staged, t.g, t.c0, p, acc,
                                                    [&](int k, int ci, const Window<-1, KWB, OFF> &win, float (&v)[KWB]) {
            const long long at = base + ci * q.SP;
            if (k == 2) win.template load<float>(gt1 + at, v);
            else win.template load<T>((k ? t1 : x) + at, v);
        });
        finish(t, pos, acc);
    }
    NDC_HD void finish(const Unit &t, long long pos, const float (&acc)[kNin][NB]) const
    {
        const long long bg = (long long)t.b * q.G + t.g;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const int i = t.c0 + c;
            if (i >= q.sc) break;
            const long long idx = (bg * q.sc + i) * q.SP + pos;
            const float n = acc[0][c] + q.eps, d = acc[1][c] + q.eps;
            const float bv = bias ? bias[t.g * q.sc + i] : 0.f, zv = Elem<T>::load(z + idx);
            if constexpr (STAGE == FWD) {
                const float s = source_of(zv, bv, q.relu);
                Elem<T>::store(out + idx, s * n / d);
                if (s_over_den) Elem<T>::store(s_over_den + idx, s / d);
                if (ratio) Elem<T>::store(ratio + idx, n / d);
            } else if constexpr (STAGE == GRAD) {
                const float inv = 1.0f / d, a = Elem<T>::load(gout + idx) * source_of(zv, bv, q.relu) * inv;
                gn[idx] = a;
                gd[idx] = -(a * n) * inv;
            } else {
                float r = Elem<T>::load(gout + idx) * n / d + acc[kNin - 1][c];
                if (q.relu && zv + bv <= 0.f) r = 0.f;   // a NaN passes, as through torch.relu's backward
                Elem<T>::store(out + idx, r);
            }
        }
    }
};

// ---------------------------------------------------------------- reductions
// A unit is one workgroup: its threads walk the positions of all samples (every nchunk-th run of
// `nt` positions), each with N sums of its own; the sums over the workgroup go to put().

// the position of a walk, advanced by a fixed step without divisions
template <typename OFF> struct Walk {
    int b;
    Pos<OFF> p;
    int sb, sd, sh, sw;
    NDC_HD Walk(const KGeom &q, long long first, long long step)
    {
        b = (int)(first / q.SP);
        p = position<OFF>(q, (OFF)(first % q.SP));
        sb = (int)(step / q.SP);
        const Pos<OFF> s = position<OFF>(q, (OFF)(step % q.SP));
        sd = s.d;
        sh = s.h;
        sw = s.w;
    }
    NDC_HD void next(const KGeom &q)
    {
        int c;
        p.w += sw;
        c = p.w >= q.W;
        p.w -= c ? q.W : 0;
        p.h += sh + c;
        c = p.h >= q.H;
        p.h -= c ? q.H : 0;
        p.d += sd + c;
        c = p.d >= q.D;
        p.d -= c ? q.D : 0;
        b += sb + c;
        p.off = ((OFF)p.d * (OFF)q.H + (OFF)p.h) * (OFF)q.W + (OFF)p.w;
    }
};

// gh[g,o,i,tau] = sum_{b,p} gt1[o,p] s[i,p+tau-pad] + gn[i,p] x[o,p+pad-tau] + gd[i,p] t1[o,p+pad-tau]
// for MB filter channels, SB source channels and KWB taps of one row
template <typename T, int MB, int SB, int KWB, typename OFF> struct FilterGrad {
    static constexpr int N = MB * SB * KWB;
    KGeom q;
    const T *x, *t1, *z;
    const float *bias, *gn, *gd, *gt1;
    float *part;                 // [chunk][stride], gh's layout
    long long stride;
    int nchunk, oblocks, iblocks, wblocks;
    struct Where {
        int chunk, tw0, th, td, i0, o0, g;
    };
    NDC_HD Where where(int u) const
    {
        Where r;
        r.chunk = u % nchunk;
        u /= nchunk;
        r.tw0 = u % wblocks * KWB;
        u /= wblocks;
        r.th = u % q.kH;
        u /= q.kH;
        r.td = u % q.kD;
        u /= q.kD;
        r.i0 = u % iblocks * SB;
        u /= iblocks;
        r.o0 = u % oblocks * MB;
        r.g = u / oblocks;
        return r;
    }
    NDC_HD void sums(int u, int tid, int nt, float (&acc)[N]) const
    {
        const Where r = where(u);
#pragma unroll
        for (int k = 0; k < N; ++k) acc[k] = 0.f;
        const long long total = (long long)q.B * q.SP, step = (long long)nchunk * nt;
        long long k = (long long)r.chunk * nt + tid;
        if (k >= total) return;
        Walk<OFF> at(q, k, step);
        for (; k < total; k += step, at.next(q)) {
            const Window<1, KWB, OFF> kwin(q, at.p, r.td, r.th, r.tw0);
            const Window<-1, KWB, OFF> awin(q, at.p, r.td, r.th, r.tw0);
            const long long bg = (long long)at.b * q.G + r.g;
            float sv[SB][KWB], nv[SB], dv[SB];
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                const int ic = r.i0 + i < q.sc ? r.i0 + i : q.sc - 1;
                const long long c = (bg * q.sc + ic) * q.SP;
                const float bv = bias ? bias[r.g * q.sc + ic] : 0.f;
                kwin.template load<T>(z + c, sv[i]);
#pragma unroll
                for (int j = 0; j < KWB; ++j) sv[i][j] = kwin.in[j] ? source_of(sv[i][j], bv, q.relu) : 0.f;
                nv[i] = load_at<float, OFF>(gn + c, at.p.off);
                dv[i] = load_at<float, OFF>(gd + c, at.p.off);
            }
#pragma unroll
            for (int o = 0; o < MB; ++o) {
                const int oc = r.o0 + o < q.m ? r.o0 + o : q.m - 1;
                const long long c = (bg * q.m + oc) * q.SP;
                float xv[KWB], tv[KWB];
                const float gv = load_at<float, OFF>(gt1 + c, at.p.off);
                awin.template load<T>(x + c, xv);
                awin.template load<T>(t1 + c, tv);
#pragma unroll
                for (int i = 0; i < SB; ++i)
#pragma unroll
                    for (int j = 0; j < KWB; ++j) {
                        float &a = acc[(o * SB + i) * KWB + j];
                        a += gv * sv[i][j];
                        a += nv[i] * xv[j];
                        a += dv[i] * tv[j];
                    }
            }
        }
    }
    NDC_HD void put(int u, int k, float v) const
    {
        const Where r = where(u);
        const int j = k % KWB, i = r.i0 + k / KWB % SB, o = r.o0 + k / KWB / SB;
        if (o >= q.m || i >= q.sc) return;
        part[r.chunk * stride + (((long long)r.g * q.m + o) * q.sc + i) * q.KT +
             (r.td * q.kH + r.th) * q.kW + r.tw0 + j] = v;
    }
};

// gb[c] = sum_{b,p} gz[b,c,p]
template <typename T> struct BiasGrad {
    static constexpr int N = 1;
    KGeom q;
    const T *gz;
    float *part;                 // [chunk][stride]
    long long stride;
    int nchunk;
    NDC_HD void sums(int u, int tid, int nt, float (&acc)[1]) const
    {
        const int chunk = u % nchunk, ch = u / nchunk;
        acc[0] = 0.f;
        const long long step = (long long)nchunk * nt;
        for (int b = 0; b < q.B; ++b) {
            const T *row = gz + ((long long)b * q.CS() + ch) * q.SP;
            for (long long p = (long long)chunk * nt + tid; p < q.SP; p += step) acc[0] += Elem<T>::load(row + p);
        }
    }
    NDC_HD void put(int u, int, float v) const { part[u % nchunk * stride + u / nchunk] = v; }
};

// ---------------------------------------------------------------- which instance

// Output channels per thread: blocks of up to 8, halved while more than half of a block would be
// padding, or while the launch has fewer than kDirectWaves wavefronts (then it is latency and not
// the load path that it waits for, and the loads of a wavefront that is more are free).
static const long long kDirectWaves = 2048;
static inline int channel_block(const KGeom &q, int cout)
{
    int nb = 8;
    while (nb > 1 && ((cout + nb - 1) / nb * nb - cout) * 2 > cout) nb /= 2;
    while (nb > 2 && (long long)q.B * q.G * ((cout + nb - 1) / nb) * ((q.SP + 63) / 64) < kDirectWaves) nb /= 2;
    return nb;
}

// Taps of a row taken at once
static inline int tap_block(const KGeom &q) { return q.kW % 3 == 0 ? 3 : q.kW % 5 == 0 ? 5 : 1; }
// 32-bit byte offsets inside a channel
static inline bool small_volume(const KGeom &q) { return q.SP < (1LL << 30); }

template <int NB, int KWB, typename OFF> struct Form {
    static constexpr int nb = NB, kwb = KWB;
    typedef OFF off;
};

// fn(Form): the instance for `cout` output channels
template <class Fn> static inline int with_form(const KGeom &q, int cout, Fn fn)
{
    if (!small_volume(q)) return fn(Form<1, 1, uint64_t>());
    const int nb = channel_block(q, cout), kwb = tap_block(q);
    if (kwb == 3)
        return nb == 8 ? fn(Form<8, 3, uint32_t>()) : nb == 4 ? fn(Form<4, 3, uint32_t>())
             : nb == 2 ? fn(Form<2, 3, uint32_t>()) : fn(Form<1, 3, uint32_t>());
    if (kwb == 5)
        return nb == 8 ? fn(Form<8, 5, uint32_t>()) : nb == 4 ? fn(Form<4, 5, uint32_t>())
             : nb == 2 ? fn(Form<2, 5, uint32_t>()) : fn(Form<1, 5, uint32_t>());
    return nb >= 4 ? fn(Form<4, 1, uint32_t>()) : fn(Form<1, 1, uint32_t>());
}

// ... for the filter gradient: MB x SB channels
template <int MB, int SB, int KWB, typename OFF> struct GradForm {
    static constexpr int mb = MB, sb = SB, kwb = KWB;
    typedef OFF off;
};
static inline int grad_block(int c) { return c >= 3 ? 4 : c == 2 ? 2 : 1; }
template <class Fn> static inline int with_grad_form(const KGeom &q, Fn fn)
{
    if (!small_volume(q)) return fn(GradForm<1, 1, 1, uint64_t>());
    const int mb = grad_block(q.m), sb = grad_block(q.sc), kwb = tap_block(q);
#define NDC_GRAD_FORM(M, S)                                                                      \
    if (mb == M && sb == S)                                                                      \
        return kwb == 3 ? fn(GradForm<M, S, 3, uint32_t>())                                      \
                        : kwb == 5 ? fn(GradForm<M, S, 5, uint32_t>()) : fn(GradForm<M, S, 1, uint32_t>())
    NDC_GRAD_FORM(1, 1);
    NDC_GRAD_FORM(1, 2);
    NDC_GRAD_FORM(1, 4);
    NDC_GRAD_FORM(2, 1);
    NDC_GRAD_FORM(2, 2);
    NDC_GRAD_FORM(2, 4);
    NDC_GRAD_FORM(4, 1);
    NDC_GRAD_FORM(4, 2);
    NDC_GRAD_FORM(4, 4);
#undef NDC_GRAD_FORM
    return NDC_ERR_GEOMETRY;
}

// Chunks the positions of a reduction are cut into: enough workgroups for two rounds of the chip,
// none with fewer than four positions a thread (its sums over the lanes would outweigh them).
static const int kReduceThreads = 256;
static inline int reduce_chunks(const KGeom &q)
{
    const int mb = small_volume(q) ? grad_block(q.m) : 1, sb = small_volume(q) ? grad_block(q.sc) : 1;
    const long long rows = q.KT / (small_volume(q) ? tap_block(q) : 1);
    const long long units = (long long)q.G * ((q.m + mb - 1) / mb) * ((q.sc + sb - 1) / sb) * rows;
    const long long most = (long long)q.B * q.SP / (kReduceThreads * 4), want = (1536 + units - 1) / units;
    const long long n = want < most ? want : most;
    return n < 1 ? 1 : (int)n;
}

}  // namespace direct
}  // namespace ndc
