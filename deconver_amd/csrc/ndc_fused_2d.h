// The NDC update of small images in one shot: depthwise k x k filters (k = 3 or 5), SC = 4.
//
// The marching kernels of ndc_fused.h walk an image row by row with two barriers a row, which is the
// cheapest way through a large launch and a chain of latencies in a small one: 32 channels of 64 x 64
// pixels gave every workgroup some sixteen row steps of 1.3 us each, on a chip that was nine tenths empty.
// Here a workgroup owns a tile of TR x TC output pixels and does everything for it at once: load with
// halo, K(s) on the tile and its halo, and the gathers -- three phases instead of sixteen steps.  The halo is
// computed again by every tile (a factor of 1.6 in K(s) for 8 x 64 pixels), which is why large launches march.
//
//   Fwd2D   out = s (A(x) + eps) / (A(K(s)) + eps), t1, and s/d, n/d where asked for
//   Bwd2D   both backward passes in one: gn, gd (from the kept s/d, n/d) on the tile and two halos,
//           gt1 = K(gd) on the tile and one halo (never stored), gx = K(gn), gz, and the sums of gh and gb
//
// A thread owns two neighbouring columns and one row of the tile (two columns and two rows of the halo tile
// in the K phases); lanes run along the columns.  Two columns, because a tap row's window of k + 1 words then
// is (k + 1) / 2 eight-byte LDS reads for 2 k products a source channel: with one column and two rows the five
// single words read for as many products took the LDS unit longer than the products the vector unit.  The
// taps are wave-uniform and come through the scalar unit, as in ndc_fused.h.  float32 arithmetic throughout, for
// bf16 storage too; gt1 is not rounded here.
#pragma once

#include "ndc_fused.h"

namespace ndc {
namespace fused {

static const int kTilePixels = 512;   // output pixels of a workgroup: two for each of 256 threads

// TC is compiled in: 32, or 16 where that covers the width with fewer columns (64 x 8 tiles have more
// halo).  Tile carries P = TC columns, TH = TR rows, ntile = tiles of an image, nseg = tiles across it, NT =
// threads, SEG = tiles a workgroup of the backward takes one after the other.
static inline bool make_tile_2d(const March &m, long long nbc, Tile &t)
{
    if (m.H != 1 || m.KH != 1 || m.KD != m.KW) return false;
    const int tc = round_up(m.W, 16) < round_up(m.W, 32) ? 16 : 32;
    int tr = kTilePixels / tc;
    if (tr > round_up(m.D, 2)) tr = round_up(m.D, 2);   // (even: the halo tiles go by pairs of rows)
    t = Tile{};
    t.P = tc;
    t.TH = tr;
    t.nseg = (m.W + tc - 1) / tc;
    t.ntile = (m.D + tr - 1) / tr * t.nseg;
    t.NT = round_up(tc * tr / 2, 64);
    // (the sums of the filter gradient over a workgroup's threads cost half as much as a tile's products: with
    // four workgroups on every CU already, a workgroup takes several tiles before it)
    const long long most = nbc * t.ntile / 1024;
    t.SEG = most < 1 ? 1 : most < t.ntile ? (int)most : t.ntile;
    return true;
}

template <int K_, int TC_> struct Tile2D {
    static constexpr int K = K_, TC = TC_, P = K / 2, SC = 4, KT = K * K, R1 = 2, NW = K + 1;
    static constexpr int SW = TC + 4 * P, XW = TC + 2 * P;   // row lengths of a tile with two halos, with one
    static NDC_HD int rows2(int TR) { return TR + 4 * P; }
    static NDC_HD int rows1(int TR) { return TR + 2 * P; }

    // the NW words of a tap row's window, from an even word
    template <class Exec> static NDC_D void window(Exec &ex, int at, float (&v)[NW])
    {
        NDC_UNROLL
        for (int u = 0; u < NW; u += 2) {
            float pair[2];
            ex.ld2(at + u, pair);
            v[u] = pair[0];
            v[u + 1] = pair[1];
        }
    }

    // K of four source planes (with a halo around the target, at `src`, `splane` words each, rows of PITCH
    // words) for N rows of two columns: row n, column c takes source rows n .. n + K - 1, columns c ..
    template <int N, int PITCH, class Exec>
    static NDC_D void scatter(Exec &ex, int src, int splane, UniformF hw, float (&acc)[N][2])
    {
        NDC_UNROLL
        for (int n = 0; n < N; ++n) acc[n][0] = acc[n][1] = 0.f;
        NDC_ROLLED
        for (int ii = 0; ii < SC; ++ii) {
            const int i = uniform_int(ii);
            float w[KT];
            load_taps<KT>(hw + i * KT, w);
            const int at = src + i * splane;
            NDC_UNROLL
            for (int q = 0; q < N + 2 * P; ++q) {
                float v[NW];
                window(ex, at + q * PITCH, v);
                NDC_UNROLL
                for (int n = 0; n < N; ++n) {
                    const int th = q - n;
                    if (th < 0 || th >= K) continue;
                    NDC_UNROLL
                    for (int tw = 0; tw < K; ++tw)
                        NDC_UNROLL
                        for (int c = 0; c < 2; ++c) acc[n][c] += v[c + tw] * w[th * K + tw];
                }
            }
        }
    }

    // A of NTEN planes (one halo around the tile) for two columns of a row; base[t]: the word
    // (own row - P, first own column - P) of plane t
    template <int NTEN, class Exec>
    static NDC_D void gather(Exec &ex, const int (&base)[NTEN], UniformF hw, float (&acc)[NTEN][SC][2])
    {
        NDC_ROLLED
        for (int thh = 0; thh < K; ++thh) {
            const int th = uniform_int(thh);
            float w[SC][K];
            load_plane_taps<SC, KT, K>(hw + th * K, w);
            NDC_UNROLL
            for (int t = 0; t < NTEN; ++t) {
                float v[NW];
                window(ex, base[t] + (2 * P - th) * XW, v);
                NDC_UNROLL
                for (int i = 0; i < SC; ++i)
                    NDC_UNROLL
                    for (int tw = 0; tw < K; ++tw)
                        NDC_UNROLL
                        for (int c = 0; c < 2; ++c) acc[t][i][c] += v[c + 2 * P - tw] * w[i][tw];
            }
        }
    }
};

// two neighbouring pixels, the second where `both`; one access where the rows allow pairs (`vec`: even
// width, aligned tensors)
template <typename T> NDC_HD void load2(const T *at, bool both, bool vec, float (&v)[2])
{
    if (vec) {
        VecIO<T, 2>::load(at, v);
    } else {
        v[0] = Elem<T>::load(at);
        v[1] = Elem<T>::load(at + (both ? 1 : 0));
    }
}
template <typename T> NDC_HD void store2(T *at, bool both, bool vec, const float (&v)[2])
{
    if (vec) {
        VecIO<T, 2>::store(at, v);
    } else {
        Elem<T>::store(at, v[0]);
        if (both) Elem<T>::store(at + 1, v[1]);
    }
}

struct Place {
    long long base;   // pixel 0 of the (sample, channel) image
    int c, r0, c0;    // channel, first row and column of the tile
};
NDC_HD Place place_2d(int bc, int tile, int C, const Tile &t, long long pixels)
{
    Place q;
    q.base = (long long)bc * pixels;
    q.c = bc % C;
    q.r0 = tile / t.nseg * t.TH;
    q.c0 = tile % t.nseg * t.P;
    return q;
}

// =================================================================== forward

template <int K_, int TC_, typename T> struct Fwd2D : Tile2D<K_, TC_> {
    typedef Tile2D<K_, TC_> B;
    static constexpr int K = K_, TC = TC_, P = B::P, SC = B::SC, KT = B::KT, R1 = B::R1, NW = B::NW, SW = B::SW, XW = B::XW;
    typedef FwdParams<T> Params;
    struct State {
    };
    static NDC_HD int lds_floats(const Tile &t) { return SC * B::rows2(t.TH) * SW + 2 * B::rows1(t.TH) * XW; }

    template <class Exec> static NDC_D void run(Exec &ex, const Params &p, int block_id)
    {
        const Tile t = p.t;
        const int TR = t.TH, RS = B::rows2(TR), RX = B::rows1(TR), H = p.D, W = p.W, nthreads = ex.nthreads;
        const long long pixels = (long long)H * W;
        const Place q = place_2d(block_id / t.ntile, block_id % t.ntile, p.C, t, pixels);
        const int off_x = SC * RS * SW, off_t = off_x + RX * XW;
        const T *xg = p.x + q.base, *zg = p.z + q.base * SC;
        T *og = p.out + q.base * SC, *t1g = p.t1 ? p.t1 + q.base : nullptr;
        UniformF hw = as_uniform(p.h + (long long)q.c * SC * KT);
        UniformF bias = as_uniform(p.bias ? p.bias + q.c * SC : p.h);
        const bool has_bias = p.bias != nullptr;
        const float floor_ = p.relu ? 0.f : pass_through_floor(), eps = p.eps;

        const bool vec = t.PL != 0;

        ex.each([&](State &, int tid) NDC_LAMBDA {
            for (int at = tid; at < RS * SW; at += nthreads) {
                const int j = at / SW, u = at - j * SW, r = q.r0 - 2 * P + j, c = q.c0 - 2 * P + u;
                const bool in = r >= 0 && r < H && c >= 0 && c < W;
                const long long px = in ? (long long)r * W + c : 0;
                float v[SC];
                NDC_UNROLL
                for (int i = 0; i < SC; ++i) v[i] = Elem<T>::load(zg + i * pixels + px);
                NDC_UNROLL
                for (int i = 0; i < SC; ++i)
                    ex.st_(i * RS * SW + at, in ? floor_f(v[i] + (has_bias ? bias[i] : 0.f), floor_) : 0.f);
            }
            for (int at = tid; at < RX * XW; at += nthreads) {
                const int j = at / XW, u = at - j * XW, r = q.r0 - P + j, c = q.c0 - P + u;
                const bool in = r >= 0 && r < H && c >= 0 && c < W;
                const float v = Elem<T>::load(xg + (in ? (long long)r * W + c : 0));
                ex.st_(off_x + at, in ? v : 0.f);
            }
        });
        ex.sync();
        // t1 = K(s) on the tile and one halo, two rows of two columns at a time
        ex.each([&](State &, int tid) NDC_LAMBDA {
            for (int at = tid; at < RX / R1 * (XW / 2); at += nthreads) {
                const int strip = at / (XW / 2), u = 2 * (at - strip * (XW / 2)), j0 = strip * R1, c = q.c0 - P + u;
                float acc[R1][2];
                B::template scatter<R1, SW>(ex, j0 * SW + u, RS * SW, hw, acc);
                NDC_UNROLL
                for (int n = 0; n < R1; ++n) {
                    const int j = j0 + n, r = q.r0 - P + j;
                    const bool in = r >= 0 && r < H;
                    const bool in0 = in && c >= 0 && c < W, in1 = in && c + 1 >= 0 && c + 1 < W;
                    const float v[2] = {in0 ? acc[n][0] : 0.f, in1 ? acc[n][1] : 0.f};
                    ex.st_(off_t + j * XW + u, v[0]);
                    ex.st_(off_t + j * XW + u + 1, v[1]);
                    // (columns go by pairs from the tile's first one on where P is even: both are the tile's)
                    if (t1g && in && j >= P && j < P + TR) {
                        if (P % 2 == 0) {
                            if (in0 && u >= P && u < P + TC) store2(t1g + (long long)r * W + c, in1, vec, v);
                        } else {
                            if (in0 && u >= P && u < P + TC) Elem<T>::store(t1g + (long long)r * W + c, v[0]);
                            if (in1 && u + 1 >= P && u + 1 < P + TC) Elem<T>::store(t1g + (long long)r * W + c + 1, v[1]);
                        }
                    }
                }
            }
        });
        ex.sync();
        ex.each([&](State &, int tid) NDC_LAMBDA {
            const int j0 = tid / (TC / 2), u = 2 * (tid - j0 * (TC / 2)), c = q.c0 + u, row = q.r0 + j0;
            if (j0 >= TR || c >= W || row >= H) return;
            float acc[2][SC][2];
            NDC_UNROLL
            for (int a = 0; a < 2; ++a)
                NDC_UNROLL
                for (int i = 0; i < SC; ++i) acc[a][i][0] = acc[a][i][1] = 0.f;
            const int ob = j0 * XW + u;
            const int base[2] = {off_x + ob, off_t + ob};
            B::template gather<2>(ex, base, hw, acc);
            const bool both = c + 1 < W;
            const long long px = (long long)row * W + c;
            NDC_UNROLL
            for (int i = 0; i < SC; ++i) {
                float s[2], o[2], rd[2], rt[2];
                ex.ld2(i * RS * SW + (j0 + 2 * P) * SW + u + 2 * P, s);
                NDC_UNROLL
                for (int e = 0; e < 2; ++e) {
                    const float inv = fast_rcp(acc[1][i][e] + eps);
                    rd[e] = s[e] * inv;
                    rt[e] = (acc[0][i][e] + eps) * inv;
                    o[e] = s[e] * rt[e];
                }
                store2(og + i * pixels + px, both, vec, o);
                if (p.s_over_den) {
                    store2(p.s_over_den + q.base * SC + i * pixels + px, both, vec, rd);
                    store2(p.ratio + q.base * SC + i * pixels + px, both, vec, rt);
                }
            }
        });
    }
};

// =================================================================== backward

template <int K_, int TC_, typename T> struct Bwd2D : Tile2D<K_, TC_> {
    typedef Tile2D<K_, TC_> B;
    static constexpr int K = K_, TC = TC_, P = B::P, SC = B::SC, KT = B::KT, R1 = B::R1, NW = B::NW, SW = B::SW, XW = B::XW;
    static constexpr int NRED = SC * KT + SC;
    typedef BwdParams<T> Params;
    struct State {
        float gacc[SC][KT], gb[SC];
    };
    static NDC_HD int lds_floats(const Tile &t)
    {
        const int main_ = SC * B::rows2(t.TH) * SW + (SC + 3) * B::rows1(t.TH) * XW, red = t.NT / 64 * NRED;
        return main_ > red ? main_ : red;
    }

    template <class Exec> static NDC_D void run(Exec &ex, const Params &p, int block_id)
    {
        const Tile t = p.t;
        const int TR = t.TH, RS = B::rows2(TR), RX = B::rows1(TR), H = p.D, W = p.W, nthreads = ex.nthreads;
        const long long pixels = (long long)H * W;
        const int groups = (t.ntile + t.SEG - 1) / t.SEG, bc = block_id / groups, group = block_id % groups;
        const Place q0 = place_2d(bc, 0, p.C, t, pixels);
        const int off_n = SC * RS * SW, off_x = off_n + SC * RX * XW, off_t = off_x + RX * XW, off_g = off_t + RX * XW;
        const T *xg = p.x + q0.base, *t1g = p.t1 + q0.base, *zg = p.z + q0.base * SC, *gg = p.gout + q0.base * SC;
        const T *dg = p.s_over_den + q0.base * SC, *rg = p.ratio + q0.base * SC;
        UniformF hw = as_uniform(p.h + (long long)q0.c * SC * KT);
        UniformF bias = as_uniform(p.bias ? p.bias + q0.c * SC : p.h);
        const bool has_bias = p.bias != nullptr;
        const float floor_ = p.relu ? 0.f : pass_through_floor();
        const int need_gh = p.need_gh;
        const bool vec = t.PL != 0;

        ex.each([&](State &st, int) NDC_LAMBDA {
            NDC_UNROLL
            for (int i = 0; i < SC; ++i) {
                st.gb[i] = 0.f;
                NDC_UNROLL
                for (int a = 0; a < KT; ++a) st.gacc[i][a] = 0.f;
            }
        });
        const int last = (group + 1) * t.SEG < t.ntile ? (group + 1) * t.SEG : t.ntile;
        for (int tt = group * t.SEG; tt < last; ++tt) {
            const Place q = place_2d(bc, uniform_int(tt), p.C, t, pixels);
            // gd on the tile and two halos, gn on the tile and one; x, t1
            ex.each([&](State &, int tid) NDC_LAMBDA {
                for (int at = tid; at < RS * SW; at += nthreads) {
                    const int j = at / SW, u = at - j * SW, r = q.r0 - 2 * P + j, c = q.c0 - 2 * P + u;
                    const bool in = r >= 0 && r < H && c >= 0 && c < W;
                    const long long px = in ? (long long)r * W + c : 0;
                    float g[SC], d[SC], n[SC];
                    NDC_UNROLL
                    for (int i = 0; i < SC; ++i) {
                        g[i] = Elem<T>::load(gg + i * pixels + px);
                        d[i] = Elem<T>::load(dg + i * pixels + px);
                        n[i] = Elem<T>::load(rg + i * pixels + px);
                    }
                    const bool inner = j >= P && j < RS - P && u >= P && u < SW - P;
                    NDC_UNROLL
                    for (int i = 0; i < SC; ++i) {
                        const float gn = in ? g[i] * d[i] : 0.f;
                        ex.st_(i * RS * SW + at, in ? -(gn * n[i]) : 0.f);
                        if (inner) ex.st_(off_n + (i * RX + j - P) * XW + u - P, gn);
                    }
                }
                for (int at = tid; at < RX * XW; at += nthreads) {
                    const int j = at / XW, u = at - j * XW, r = q.r0 - P + j, c = q.c0 - P + u;
                    const bool in = r >= 0 && r < H && c >= 0 && c < W;
                    const long long px = in ? (long long)r * W + c : 0;
                    const float vx = Elem<T>::load(xg + px), vt = Elem<T>::load(t1g + px);
                    ex.st_(off_x + at, in ? vx : 0.f);
                    ex.st_(off_t + at, in ? vt : 0.f);
                }
            });
            ex.sync();
            ex.each([&](State &st, int tid) NDC_LAMBDA {
                for (int at = tid; at < RX / R1 * (XW / 2); at += nthreads) {   // gt1 = K(gd), as t1 in the forward
                    const int strip = at / (XW / 2), u = 2 * (at - strip * (XW / 2)), j0 = strip * R1, c = q.c0 - P + u;
                    float acc[R1][2];
                    B::template scatter<R1, SW>(ex, j0 * SW + u, RS * SW, hw, acc);
                    NDC_UNROLL
                    for (int n = 0; n < R1; ++n) {
                        const int r = q.r0 - P + j0 + n;
                        const bool in = r >= 0 && r < H;
                        ex.st_(off_g + (j0 + n) * XW + u, in && c >= 0 && c < W ? acc[n][0] : 0.f);
                        ex.st_(off_g + (j0 + n) * XW + u + 1, in && c + 1 >= 0 && c + 1 < W ? acc[n][1] : 0.f);
                    }
                }
                const int j0 = tid / (TC / 2), u = 2 * (tid - j0 * (TC / 2)), c = q.c0 + u, row = q.r0 + j0;
                if (j0 >= TR || c >= W || row >= H) return;
                const int ob = j0 * XW + u;
                if (p.gx) {
                    float acc[1][2];
                    B::template scatter<1, XW>(ex, off_n + ob, RX * XW, hw, acc);
                    store2(p.gx + q.base + (long long)row * W + c, c + 1 < W, vec, acc[0]);
                }
                if (need_gh) {
                    // (gn, gd of a second column past the image are zeros; its products with x and t1 past the
                    // image are left out, so that nothing but zeros is ever added for it)
                    float gn[SC][2], gd[SC][2];
                    NDC_UNROLL
                    for (int i = 0; i < SC; ++i) {
                        NDC_UNROLL
                        for (int e = 0; e < 2; ++e) gn[i][e] = ex.ld(off_n + (i * RX + j0 + P) * XW + u + P + e);
                        ex.ld2((i * RS + j0 + 2 * P) * SW + u + 2 * P, gd[i]);
                    }
                    const bool both = c + 1 < W;
                    NDC_UNROLL
                    for (int th = 0; th < K; ++th) {
                        float vx[NW], vt[NW];
                        B::window(ex, off_x + ob + (2 * P - th) * XW, vx);
                        B::window(ex, off_t + ob + (2 * P - th) * XW, vt);
                        NDC_UNROLL
                        for (int i = 0; i < SC; ++i)
                            NDC_UNROLL
                            for (int tw = 0; tw < K; ++tw) {
                                float a = st.gacc[i][th * K + tw];
                                a += gn[i][0] * vx[2 * P - tw];
                                a += gd[i][0] * vt[2 * P - tw];
                                a += gn[i][1] * (both ? vx[1 + 2 * P - tw] : 0.f);
                                a += gd[i][1] * (both ? vt[1 + 2 * P - tw] : 0.f);
                                st.gacc[i][th * K + tw] = a;
                            }
                    }
                }
            });
            ex.sync();
            ex.each([&](State &st, int tid) NDC_LAMBDA {
                const int j0 = tid / (TC / 2), u = 2 * (tid - j0 * (TC / 2)), c = q.c0 + u, row = q.r0 + j0;
                if (j0 >= TR || c >= W || row >= H) return;
                const int ob = j0 * XW + u;
                const bool both = c + 1 < W;
                const long long px = (long long)row * W + c;
                float s[SC][2], acc[1][SC][2];
                NDC_UNROLL
                for (int i = 0; i < SC; ++i) {
                    float g[2], r[2];
                    load2(zg + i * pixels + px, both, vec, s[i]);
                    load2(gg + i * pixels + px, both, vec, g);
                    load2(rg + i * pixels + px, both, vec, r);
                    acc[0][i][0] = g[0] * r[0];
                    acc[0][i][1] = g[1] * r[1];
                }
                const int base[1] = {off_g + ob};
                B::template gather<1>(ex, base, hw, acc);
                NDC_UNROLL
                for (int i = 0; i < SC; ++i) {
                    float gz[2];
                    NDC_UNROLL
                    for (int e = 0; e < 2; ++e) {
                        s[i][e] = floor_f(s[i][e] + (has_bias ? bias[i] : 0.f), floor_);
                        gz[e] = acc[0][i][e];
                        if (p.relu && s[i][e] <= 0.f) gz[e] = 0.f;   // a NaN passes
                    }
                    st.gb[i] += gz[0] + (both ? gz[1] : 0.f);
                    if (p.gz) store2(p.gz + q.base * SC + i * pixels + px, both, vec, gz);
                    if (!both) s[i][1] = 0.f;
                }
                if (need_gh) {
                    NDC_UNROLL
                    for (int th = 0; th < K; ++th) {
                        float v[NW];
                        B::window(ex, off_g + ob + (2 * P - th) * XW, v);
                        NDC_UNROLL
                        for (int i = 0; i < SC; ++i)
                            NDC_UNROLL
                            for (int tw = 0; tw < K; ++tw) {
                                float a = st.gacc[i][th * K + tw];
                                a += s[i][0] * v[2 * P - tw];
                                a += s[i][1] * (both ? v[1 + 2 * P - tw] : 0.f);
                                st.gacc[i][th * K + tw] = a;
                            }
                    }
                }
            });
            ex.sync();   // (the tile's LDS is the next one's)
        }
        if (p.need_gh || p.need_gb) {
            float *dst = p.part + (long long)block_id * p.part_stride;
            ex.template block_reduce<NRED>(
                [](State &st, int i) NDC_LAMBDA {
                    return i < SC * KT ? st.gacc[(i < SC * KT ? i : 0) / KT][i % KT] : st.gb[i >= SC * KT ? i - SC * KT : 0];
                },
                [&](int i, float v) NDC_LAMBDA { dst[i] = v; });
        }
    }
};

}  // namespace fused
}  // namespace ndc
