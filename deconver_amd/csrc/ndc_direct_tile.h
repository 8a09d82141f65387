// The direct kernels' convolutions from boxes in LDS: filters of 3 x 3 or 5 x 5 taps in the last two axes (any number
// in the first), the functors of ndc_direct.h.
//
// A workgroup makes a box of positions for one unit (sample, group, block of output channels), a thread one position or
// two of neighbouring rows.  It stages the box with its halo, zeros outside the volume, for as many input channels as
// its LDS share takes, and those channels' weights in the order they are used; then every thread runs over channels and
// taps without a bounds check, an address or a load from memory, both factors of a product in vector registers (3.3
// clocks a multiply-add, 4.4 with one in a scalar register).  Two rows a thread share the weights of a row and the
// window rows between them.  Without boxes a thread waits for the loads of every tap row, some twenty round trips to the
// L2 in a row, which is what small launches spent their time on; here it is one round trip per group of channels.
// What bounds them now: the multiply-adds of large launches; in small ones the launch, that round trip, the products of
// the one or two wavefronts a SIMD has and the epilogue follow each other.
// us, one position at a time (ndc_direct.h) -> boxes, float32: 4 groups of 4 and 8 channels on 2 x 24^3, t1 30 -> 22,
// the forward's ratio 26 -> 17, gn and gd 26 -> 17, gx and gt1 25 -> 23, gz 36 -> 23; forward and backward in all
// 194 -> 154 (the layer's call 206 -> 166), 2 groups with 5^3 taps on 12 x 13 x 15 438 -> 247, 16 channels 1 -> 2 on 2 x 24^3 122 -> 94, 64 channels
// 1 -> 2 with 5 x 5 taps on 4 x 128^2 618 -> 452, 16 groups of 4 and 8 on 2 x 48 x 50 x 46 2838 -> 2538; behind in none of
// 19 layers measured (0.56 to 0.93 of the time).
#pragma once

#include "ndc_direct.h"
#include "ndc_exec.h"

#include <cstring>

namespace ndc {
namespace direct {

struct Box {
    int NR;                  // rows of positions a thread makes, 1 or 2
    int TD, TH, TW, HP;      // positions of a workgroup, and how many threads share their rows of a plane
    int SD, SH, SW, SV;      // staged extents and their product
    int nd, nh, nw, tiles;   // boxes per axis and volume
    int chunk;               // input channels staged at once
    int NT;                  // threads of a workgroup
    uint32_t over_sw, over_sh;   // 2^32 / SW and 2^32 / SH, rounded up (see quotient)
};

// v / d from o = 2^32 / d rounded up: exact while v * d < 2^32 (d > 1), and staged extents are below 2^16
static NDC_HD int quotient(int v, uint32_t o) { return (int)(((uint64_t)(uint32_t)v * o) >> 32); }

static NDC_HD int box_weights(const KGeom &q, int nb) { return q.KT * nb; }
// words of LDS: the staged channels of the inputs, the weights from a multiple of four words on
static NDC_HD int box_values(const Box &t, int nin) { return (nin * t.chunk * t.SV + 3) / 4 * 4; }

template <class F, int K, int NR> struct Tiled {
    static constexpr int NIN = F::kNin, NB = F::kNB, ROW = NB * K;
    static_assert(F::kKWB == K, "a tap row at a time");
    struct Params {
        F f;
        Box t;
    };
    struct State {
        float acc[NR][NIN][NB];
        int at, pos, live, live1;
    };
    static int lds_floats(const KGeom &q, const Box &t) { return box_values(t, NIN) + t.chunk * box_weights(q, NB); }

    template <class Exec> static NDC_D void run(Exec &ex, const Params &p, int block)
    {
        const F &f = p.f;
        const Box t = p.t;
        const KGeom &q = f.q;
        const int u = block / t.tiles, tile = block - u * t.tiles;
        const int iw = tile % t.nw, r0 = tile / t.nw, d0 = r0 / t.nh * t.TD, h0 = r0 % t.nh * t.TH, w0 = iw * t.TW;
        const Unit un(u, q.G, f.blocks, NB);
        const int cin = F::kAdj ? q.m : q.sc, cout = F::kAdj ? q.sc : q.m, rows = q.kD * K, wbase = box_values(t, NIN);
        const float *hg = f.hf + (long long)un.g * q.m * q.sc * q.KT;

        ex.each([&](State &st, int tid) NDC_LAMBDA {
            const int w = tid % t.TW, r = tid / t.TW, h = r % t.HP * NR, d = r / t.HP;
            st.live = d < t.TD && d0 + d < q.D && h0 + h < q.H && w0 + w < q.W;
            st.live1 = st.live && h + 1 < t.TH && h0 + h + 1 < q.H;
            st.at = (d * t.SH + h) * t.SW + w;
            st.pos = ((d0 + d) * q.H + h0 + h) * q.W + w0 + w;
#pragma unroll
            for (int n = 0; n < NR; ++n)
#pragma unroll
                for (int k = 0; k < NIN; ++k)
#pragma unroll
                    for (int c = 0; c < NB; ++c) st.acc[n][k][c] = 0.f;
        });
        for (int c0 = 0; c0 < cin; c0 += t.chunk) {
            const int nc = cin - c0 < t.chunk ? cin - c0 : t.chunk;
            if (c0) ex.sync();
            ex.each([&](State &, int tid) NDC_LAMBDA {
                for (int e = tid; e < t.SV; e += t.NT) {
                    const int r = quotient(e, t.over_sw), d = quotient(r, t.over_sh);
                    const int dd = d0 + d - q.pD, hh = h0 + r - d * t.SH - q.pH, ww = w0 + e - r * t.SW - q.pW;
                    const bool in = (unsigned)dd < (unsigned)q.D && (unsigned)hh < (unsigned)q.H && (unsigned)ww < (unsigned)q.W;
                    const uint32_t off = in ? ((uint32_t)dd * q.H + hh) * q.W + ww : 0u;
#pragma unroll 4
                    for (int ci = 0; ci < nc; ++ci)
#pragma unroll
                        for (int k = 0; k < NIN; ++k) {
                            const float v = f.value(k, un, c0 + ci, off);
                            ex.st_((k * t.chunk + ci) * t.SV + e, in ? v : 0.f);
                        }
                }
                // weights: [input channel][tap row][output channel][K]; channels past the last repeat the last
                for (int e = tid; e < nc * rows; e += t.NT) {
                    float w[ROW];
                    load_weights(q, hg, un, cout, rows, c0, e, w);
#pragma unroll
                    for (int i = 0; i < ROW; ++i) ex.st_(wbase + e * ROW + i, w[i]);
                }
            });
            ex.sync();
            ex.each([&](State &st, int) NDC_LAMBDA {
                if (!st.live) return;
                for (int ci = 0; ci < nc; ++ci)
                    for (int td = 0; td < q.kD; ++td) {
                        // (A takes the taps from the far end of the window)
                        const int sd = F::kAdj ? q.kD - 1 - td : td;
                        const int wrow = wbase + (ci * q.kD + td) * K * ROW;
                        float w[NR][ROW];   // row s of the window meets tap rows s, s - 1 of the positions' NR rows
#pragma unroll
                        for (int s = 0; s < K + NR - 1; ++s) {
                            float v[NIN][K];
                            if (s < K) row_words(ex, wrow + (F::kAdj ? K - 1 - s : s) * ROW, w[s % NR]);
#pragma unroll
                            for (int k = 0; k < NIN; ++k) {
                                const int from = st.at + ((k * t.chunk + ci) * t.SV + (sd * t.SH + s) * t.SW);
#pragma unroll
                                for (int j = 0; j < K; ++j) v[k][F::kAdj ? K - 1 - j : j] = ex.ld(from + j);
                            }
#pragma unroll
                            for (int n = 0; n < NR; ++n) {
                                if (s - n < 0 || s - n >= K) continue;
#pragma unroll
                                for (int c = 0; c < NB; ++c)
#pragma unroll
                                    for (int j = 0; j < K; ++j)
#pragma unroll
                                        for (int k = 0; k < NIN; ++k) st.acc[n][k][c] += v[k][j] * w[(s - n) % NR][c * K + j];
                            }
                        }
                    }
            });
        }
        ex.each([&](State &st, int) NDC_LAMBDA {
            if (st.live) f.finish(un, st.pos, st.acc[0]);
            if (NR > 1 && st.live1) f.finish(un, st.pos + q.W, st.acc[NR - 1]);
        });
    }

    static NDC_HD void load_weights(const KGeom &q, const float *hg, const Unit &un, int cout, int rows, int c0, int e, float (&w)[ROW])
    {
        const int ci = e / rows, row = e - ci * rows;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const int k = un.c0 + c < cout ? un.c0 + c : cout - 1;
#pragma unroll
            for (int j = 0; j < K; ++j)
                w[c * K + j] = hg[((F::kAdj ? c0 + ci : k) * q.sc + (F::kAdj ? k : c0 + ci)) * q.KT + row * K + j];
        }
    }

    // a row of weights (from a multiple of four words where it is that long)
    template <class Exec> static NDC_D void row_words(Exec &ex, int at, float (&w)[ROW])
    {
        if constexpr (ROW % 4 == 0) {
#pragma unroll
            for (int i = 0; i < ROW; i += 4) {
                uint32_t v[4];
                ex.ld4a(at + i, v);
#pragma unroll
                for (int j = 0; j < 4; ++j) w[i + j] = bits_to_float(v[j]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < ROW; ++i) w[i] = ex.ld(at + i);
        }
    }
};

#ifndef NDC_BOX_WEIGHED
#define NDC_BOX_WEIGHED()   // (the host build counts the boxes it looks at)
#endif
// The box of a launch: the least cost over one or two rows a thread and the boxes that cut an axis into equal parts, of the
// first axis at most 32, of the second 16, of the last 6.  Volumes of which such parts have more than 512 threads' positions
// (144^3 and 320^2, not 128^3 and 256^2) have no box.
// The cost is what the busiest CU has to do: products and LDS reads of its SIMDs (dearer where a SIMD has fewer than two
// wavefronts), the values and 128-byte lines staged, the lines its outputs touch, and a fixed part for every round of
// workgroups the CU holds at once times the groups of channels.  Its constants were fitted to 70 boxes each of five
// kernels on seven layers, on which the box it takes is 5 % behind the best one (a box for the most threads alone: 16 %).
static inline bool choose_box(const KGeom &q, int nin, int nb, int cin, long long units, Box &best)
{
    const int K = q.kW, weights = box_weights(q, nb), budget = 10 * 1024, kMaxLds = 160 * 1024;
    double least = 0;
    best.NT = 0;
    // the extents that equal parts of an axis have, and how many of them it takes
    struct Parts {
        int n = 0, extent[32], count[32];
        Parts(int of, int most)
        {
            for (int p = 1; p <= most && p <= of; ++p) {
                const int e = (of + p - 1) / p;
                if (n && extent[n - 1] == e) continue;
                extent[n] = e, count[n++] = (of + e - 1) / e;
            }
        }
    };
    const Parts pw(q.W, 6), ph(q.H, 16), pd(q.D, 32);
    auto row_cost = [&](double product, int nr) { return product * nr * nb * K * nin + 0.8 * nb * K + 0.75 * nin * (K + nr - 1); };
    for (int nr = 1; nr <= 2; ++nr) {
        // wavefronts a SIMD has the registers for
        int simd = 512 / (46 + nr * nb * (nin + K) + 2 * nin * K);
        simd = simd < 1 ? 1 : simd > 8 ? 8 : simd;
        const double least_row = row_cost(1.1, nr);
        for (int iw = 0; iw < pw.n; ++iw)
            for (int ih = 0; ih < ph.n; ++ih) {
                Box t;
                t.NR = nr, t.TW = pw.extent[iw], t.TH = ph.extent[ih], t.HP = (t.TH + nr - 1) / nr;
                t.SH = t.HP * nr + K - 1, t.SW = t.TW + K - 1, t.nh = ph.count[ih], t.nw = pw.count[iw];
                if (t.TW > 512 || t.HP > 512) continue;
                for (int id = 0; id < pd.n; ++id) {
                    t.TD = pd.extent[id], t.nd = pd.count[id], t.tiles = t.nd * t.nh * t.nw;
                    const long long n = (long long)t.TW * t.HP * t.TD;
                    if (n > 512) continue;
                    NDC_BOX_WEIGHED();
                    t.NT = (int)((n + 63) / 64 * 64);
                    t.SD = t.TD + q.kD - 1, t.SV = t.SD * t.SH * t.SW;
                    const int words = nin * t.SV + weights;   // of a channel
                    if (words > budget) continue;
                    const long long group = (units * t.tiles + 255) / 256;   // workgroups of the busiest CU
                    const int w = t.NT / 64;
                    const double rows = (double)((group * w + 3) / 4) * cin * (q.KT / K);
                    const double staging = (double)group * cin * nin * (t.SV / 64.0 * 8 + 8.4 * t.SD * t.SH * (t.SW / 32.0 + 1));
                    const double out = group * 40.0 * nb * t.TD * t.TH * (t.TW / 32.0 + 1);
                    if (best.NT) {
                        // the least that it can cost, without the divisions: as many workgroups a CU as registers allow
                        const double share = w / (4.0 * simd), rounds = group * (share < 1 ? share : 1.0), groups = cin * (double)words * (1.0 / budget);
                        const double fixed = (rounds > 1 ? rounds : 1.0) * (groups > 1 ? groups : 1.0) * 40e3;
                        if ((rows * least_row + 0.66 * staging + out + fixed) * (1 - 1e-9) > least) {
                            if (n < 64) break;
                            continue;
                        }
                    }
                    t.chunk = budget / words;
                    if (t.chunk > cin) t.chunk = cin;
                    int held = kMaxLds / (4 * t.chunk * words);   // workgroups a CU has the place for
                    if (held * w > 4 * simd) held = 4 * simd / w;
                    if (held > group) held = (int)group;
                    if (held < 1) held = 1;
                    const double per_simd = held * w / 4.0, product = per_simd >= 2 ? 1.1 : 1.1 * (1 + 0.37 * (2 - (per_simd < 1 ? 1 : per_simd)));
                    const double cost = rows * row_cost(product, nr) + (held == 1 ? 1.0 : 0.66) * staging + out +
                                        (double)((group + held - 1) / held) * ((cin + t.chunk - 1) / t.chunk) * 40e3;
                    if (!best.NT || cost < least) best = t, least = cost;
                    if (n < 64) break;
                }
            }
    }
    if (!best.NT) return false;
    best.over_sw = 0xffffffffu / best.SW + 1, best.over_sh = 0xffffffffu / best.SH + 1;
    return true;
}

// ... of the sizes a thread saw last.  A search takes the host 2 to 8 us, and a layer with its backward asks for five: what
// is kept serves some hundred sizes, so that a network searches once.
static inline bool box_of(const KGeom &q, int nin, int nb, int cin, long long units, Box &box)
{
    if ((q.kW != 3 && q.kW != 5) || q.kH != q.kW || !small_volume(q) || tap_block(q) != q.kW) return false;
    static const int kWords = 10, kEntries = 1024, kWays = 4;
    struct Entry {
        int key[kWords];   // zeros where nothing is kept (a filter has kW > 0)
        bool ok;
        Box box;
    };
    static thread_local Entry kept[kEntries] = {};
    static thread_local unsigned turn = 0;
    const int key[kWords] = {q.kW, q.kD, q.D, q.H, q.W, nin, nb, cin, (int)(units >> 32), (int)units};
    unsigned at = 0;
    for (int k : key) at = ((at ^ at >> 15) + (unsigned)k) * 0x9e3779b1u;
    Entry *set = kept + (at >> 16) % (kEntries / kWays) * kWays;
    int way = 0;
    for (; way < kWays && set[way].key[0]; ++way)
        if (!memcmp(set[way].key, key, sizeof(key))) {
            box = set[way].box;
            return set[way].ok;
        }
    Entry &e = set[way < kWays ? way : (int)(turn++ % kWays)];
    e.ok = choose_box(q, nin, nb, cin, units, e.box);
    memcpy(e.key, key, sizeof(key));
    box = e.box;
    return e.ok;
}

// ... if a launch takes them: fewer than 2^32 threads (46 x 1 x 60 positions are six boxes of 512 threads a unit where they
// were 2816 threads one position at a time)
static inline bool takes_boxes(const KGeom &q, int nin, int nb, int cin, long long units, Box &box)
{
    return box_of(q, nin, nb, cin, units, box) && units * box.tiles < (1LL << 31) && units * box.tiles * box.NT < (1LL << 32);
}

template <class BE, class F, int K, int NR> static int launch_boxes(const F &f, const Box &t, long long units, void *stream)
{
    typedef Tiled<F, K, NR> Kernel;
    const typename Kernel::Params p = {f, t};
    return BE::template block_kernel<Kernel>(p, (int)(units * t.tiles), t.NT, Kernel::lds_floats(f.q, t), stream);
}

// a functor over all its units and positions: from tiles where its filter is of that form
template <class BE, class F> static int launch(const F &f, long long units, void *stream)
{
    if constexpr (F::kKWB == 3 || F::kKWB == 5) {
        constexpr int K = F::kKWB;
        Box t;
        if (takes_boxes(f.q, F::kNin, F::kNB, F::kAdj ? f.q.m : f.q.sc, units, t))
            return t.NR == 2 ? launch_boxes<BE, F, K, 2>(f, t, units, stream) : launch_boxes<BE, F, K, 1>(f, t, units, stream);
    }
    return BE::weighted_unit(units, f.q.SP, stream, f);
}

}  // namespace direct
}  // namespace ndc
