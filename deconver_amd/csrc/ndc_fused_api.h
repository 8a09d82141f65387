// Host side of the fused kernels: which geometries they cover, launch shapes, scratch
// layout, and the launch sequence of a forward / backward call.  Needs a `Backend` with
// `block_kernel<Kernel>(params, nblocks, nthreads, lds_floats, stream)` and `elementwise`.
#pragma once

#include "../../include/deconver_ndc.h"
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <type_traits>

#include "ndc_fused.h"
#include "ndc_fused_mfma.h"
#include "ndc_fused_2d.h"

namespace ndc {
namespace fused {

// Compiled instances, in the marching view (2-D k x k runs as (k, 1, k)).  One row per
// (KD, KH, KW, SC, RHF, RWF, RHB, RWB): RHF x RWF is the register tile (rows x columns per
// thread) of the forward kernel, RHB x RWB that of the two backward kernels.  Rows of one
// filter geometry are listed in order of preference; a row with RW = 2 needs an even W and
// tensors aligned to two elements; RW = -2 is the same for any width and alignment; every geometry also has
// an RW = 1 row.
#define NDC_FUSED_VARIANTS(X)        \
    X(3, 3, 3, 4, 2, 2, 2, 2)        \
    X(3, 3, 3, 4, 2, 2, 1, 2)        \
    X(3, 3, 3, 4, 2, -2, 2, -2)      \
    X(3, 3, 3, 4, 2, -2, 2, 1)       \
    X(3, 3, 3, 4, 4, 1, 2, -2)       \
    X(3, 3, 3, 4, 4, 1, 2, 1)        \
    X(3, 3, 3, 4, 2, 1, 1, 1)        \
    X(5, 1, 5, 4, 1, 2, 1, 2)        \
    X(5, 1, 5, 4, 1, -2, 1, -2)      \
    X(5, 1, 5, 4, 1, -2, 1, 1)       \
    X(5, 1, 5, 4, 1, 1, 1, -2)       \
    X(5, 1, 5, 4, 1, 1, 1, 1)        \
    X(3, 1, 3, 4, 1, 2, 1, 2)        \
    X(3, 1, 3, 4, 1, -2, 1, -2)      \
    X(3, 1, 3, 4, 1, -2, 1, 1)       \
    X(3, 1, 3, 4, 1, 1, 1, -2)       \
    X(3, 1, 3, 4, 1, 1, 1, 1)

// What a plan may use: one column a thread; in the forward also pairs at any width and alignment; in the backward
// too; pairs of aligned tensors of an even width.
enum { kSingles = 0, kLooseForward = 1, kLoosePairs = 2, kPairs = 3 };

struct Variant {
    int KD, KH, KW, SC, RHF, RWF, RHB, RWB;
};

// Launch-shape choices that are not dictated by the geometry: the measured best, fixed at
// compile time.  A tuning build (-DNDC_TUNING, never the shipped library) reads them from
// NDC_TUNE_* environment variables once, at the first call.
struct Tuning {
    int rhf, rwf, rhb, rwb;      // forced register tiles (0: the table's order of preference)
    int threads_f, threads_b;    // workgroup sizes of the FMA kernels, forward / backward
    int threads_f2, threads_b2;  // ... of the bf16 dot2 kernels, and the other size tried by cost_tile
    int threads_f2_wide, threads_b2_narrow;
    int split, dot2;             // march segments on / bf16 dot2 kernels on
    int mfma;                    // bf16 matrix-instruction kernels on (where they cover the geometry)
};

#ifdef NDC_TUNING
static inline int env_int(const char *name, int dflt)
{
    const char *v = getenv(name);
    return v && *v ? atoi(v) : dflt;
}
static inline const Tuning &tuning()
{
    static const Tuning t = {env_int("NDC_TUNE_RHF", 0),  env_int("NDC_TUNE_RWF", 0),
                             env_int("NDC_TUNE_RHB", 0),  env_int("NDC_TUNE_RWB", 0),
                             env_int("NDC_TUNE_NTF", 256), env_int("NDC_TUNE_NTB", 512),
                             env_int("NDC_TUNE_NTF2", 256), env_int("NDC_TUNE_NTB2", 256),
                             env_int("NDC_TUNE_NTF2W", 512), env_int("NDC_TUNE_NTB2N", 128),
                             env_int("NDC_TUNE_SPLIT", 1), env_int("NDC_TUNE_DOT2", 1),
                             env_int("NDC_TUNE_MFMA", 1)};
    return t;
}
#else
static inline Tuning tuning() { return Tuning{0, 0, 0, 0, 256, 512, 256, 256, 512, 128, 1, 1, 1}; }
#endif

// where column pairs of rows of any length and alignment are taken (see loose_pairs)
struct LoosePairs {
    bool forward, backward;
};

// first listed row of this filter geometry that the width / alignment allow (and, in a
// tuning run, that matches the requested register tiles)
static inline bool find_variant(const KGeom &q, const March &m, int pairs, const LoosePairs &loose, Variant &v)
{
    if (q.m != 1) return false;
    const Tuning tn = tuning();
    // 2-D problems march along the image rows with one strip of lanes across a row: below
    // 128 columns a lane per column (not per column pair) keeps more of the wavefront busy
    // (measured 16-32 % faster from 16 to 100 columns, 4-15 % slower from 128 on)
    const bool narrow_2d = m.H == 1 && m.W < 128 && !tn.rwf && !tn.rwb;
    const bool even = pairs == kPairs && m.W % 2 == 0 && !narrow_2d;
    const bool loose_f = pairs >= kLooseForward && loose.forward, loose_b = pairs >= kLoosePairs && loose.backward;
    auto takes = [&](int rwf, int rwb) {
        return (rwf == 1 || (rwf == 2 ? even : loose_f)) && (rwb == 1 || (rwb == 2 ? even : loose_b));
    };
    bool found = false;
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                        \
    if (!found && m.KD == kd_ && m.KH == kh_ && m.KW == kw_ && q.sc == sc_ &&                \
        takes(rwf_, rwb_) && (!tn.rhf || tn.rhf == rhf_) &&                 \
        (!tn.rwf || tn.rwf == rwf_) && (!tn.rhb || tn.rhb == rhb_) &&                        \
        (!tn.rwb || tn.rwb == rwb_)) {                                                       \
        v = Variant{kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_};                             \
        found = true;                                                                        \
    }
    NDC_FUSED_VARIANTS(X)
#undef X
    if (found) return true;
    // no row matches a tuning request: fall back to the plain order of preference
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                        \
    if (!found && m.KD == kd_ && m.KH == kh_ && m.KW == kw_ && q.sc == sc_ &&                \
        takes(rwf_, rwb_)) {                                                \
        v = Variant{kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_};                             \
        found = true;                                                                        \
    }
    NDC_FUSED_VARIANTS(X)
#undef X
    return found;
}

// The process-wide default of the kernel family for calls that do not name one
// (ndc_matrix_kernels): 0 = vector unit, 1 = the kernels built on the 4x4x4 matrix instruction
// (ndc_fused_mfma.h) where they cover the geometry.  Off unless a caller turns it on: the path
// is specified as a depthwise stencil that keeps matrix instructions out of it.  Atomic, so
// that a thread that sets it and threads that launch do not race; a call that must not depend
// on it names its family in ndc_geom.path.
static inline std::atomic<int> &matrix_default()
{
    static std::atomic<int> on{0};
    return on;
}

#ifndef NDC_SPLIT_F
#define NDC_SPLIT_F 4096
#endif
#ifndef NDC_SPLIT_B
#define NDC_SPLIT_B 2048
#endif
static const long long kSplitWavesF = NDC_SPLIT_F, kSplitWavesB = NDC_SPLIT_B;

// 2-D problems of up to so many pixels in all, and of small images up to so many, run tile by tile
// (ndc_fused_2d.h), forward and backward.  us marching -> in tiles, 5x5, float32 (bf16 within 10 %):
//   forward   32 x 64^2 18 -> 8, 512 x 8^2 21 -> 8, 32 x 128^2 36 -> 17, 64 x 104 x 88 25 -> 21, 2 x 32 x 150 x 170
//             (1.6 M) 59 -> 46, 8 x 256 x 32^2 (2.1 M) 76 -> 41; 8 x 128 x 64^2 (4.2 M) 85 -> 85, 8 x 64 x 128^2 129 -> 164
//   backward  32 x 64^2 48 -> 20, 512 x 13 x 11 73 -> 21, 32 x 128^2 67 -> 49, 4 x 64 x 50 x 70 (0.9 M) 87 -> 84,
//             8 x 256 x 32^2 (2.1 M) 148 -> 101; 32 x 208 x 176 (1.2 M) 89 -> 95, 8 x 128 x 64^2 175 -> 235
// A tile costs the same where it is part empty, so the pixels that tiles cover count too, and a march costs whole
// wavefronts across a row.  5x5: 8 x 281 x 33 x 34 covers 6.9 M pixels and took 92 -> 112 forward, 8 x 129 x 43 x 66
// 5.3 M and 111 -> 94.  3x3 marches on fewer products a pixel: tiles up to 0.85 M covered pixels forward and 0.65 M
// backward, or where they cover clearly fewer than the march has lanes.  us, 3x3, float32, marching -> tiles, with
// covered pixels / lanes:
//   forward             80 x 80 x 83 (0.61 M) 19 -> 13, 8 x 49 x 27 x 49 (0.80 M) 17.6 -> 14.0, 8 x 662 x 13 x 17
//                       (2.4 / 4.4 M) 48 -> 30, 8 x 35 x 58 x 65 (1.4 / 2.1 M) 33 -> 27, 8 x 126 x 51 x 58 (4.1 / 3.3 M) 42 -> 56
//   forward + backward  184 x 41 x 34 (0.57 M) 46 -> 45, 8 x 91 x 19 x 33 (0.70 / 0.89 M) 63 -> 68,
//                       8 x 64 x 33 x 33 (1.6 / 1.1 M) 67 -> 81, 8 x 213 x 27 x 34 (2.3 / 2.9 M) 108 -> 143
static const long long kPixelsF = 1700 * 1000, kSmallImagesF = 3000 * 1000, kCoveredF = 5500 * 1000;
static const long long kPixelsB = 900 * 1000, kSmallImagesB = 2500 * 1000;
static const long long kCovered3F = 850 * 1000, kCovered3B = 650 * 1000;

// (0 in a host build whose tests send every image down the march)
#ifndef NDC_TILES_2D
#define NDC_TILES_2D 1
#endif

struct Plan {
    Variant v;
    March m;
    bool dot2;            // bf16 dot2 kernels (3x3x3, SC = 4, even W, aligned pairs)
    bool mfma1, mfma2;    // ... with pass 1 / pass 2 on the matrix instruction when they read the forward's ratios
    bool mfmaf;           // ... with the forward on the matrix instruction
    bool small_f, small_b;   // one-shot kernels of small images (ndc_fused_2d.h); the backward where it has the ratios
    Tile t2;                 // ... their tiles
    int nblk_f2, nblk_b2;
    Tile tf, tb;          // forward / backward launch shapes
    int lds_f, lds_b1, lds_b2;
    int nblk_f, nblk_b;
};

#define NDC_IS_VARIANT(pl, kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                          \
    ((pl).v.KD == kd_ && (pl).v.KH == kh_ && (pl).v.KW == kw_ && (pl).v.SC == sc_ &&            \
     (pl).v.RHF == rhf_ && (pl).v.RWF == rwf_ && (pl).v.RHB == rhb_ && (pl).v.RWB == rwb_)

// What a launch of the 3-D kernels takes, up to a factor: the wavefronts a SIMD of the
// busiest CU works through, times the planes a workgroup marches over.
//   * R workgroups of a CU run at once (LDS and registers; a workgroup's wavefronts go round the
//     four SIMDs, so six count as eight).  q resident ones take q ceil(w / 4) + `alone`: a SIMD with
//     one wavefront waits for half of its time (1) or more, with four hardly ever.
//   * a segment of the march adds the planes its neighbours own (3 more than it keeps), a row band
//     the two halo rows it computes twice (a fifth of a strip's work each).
//   * behind full rounds a remainder runs into the round before it: `overlap` of it costs its share of
//     a full round, the rest a round of its own.
//   * `mixed`: from two full rounds on, workgroups of different rounds overlap and a remainder
//     costs its share only (the dot2 forward, whose four wavefronts per SIMD drift apart).
// bf16 dot2 kernels: against the best of 56 launch shapes measured on each of 22 problems (16^3 ..
// 192^3, widths 14 to 192, 32 to 512 channels) the choice is 1 % behind on average and 11 % at worst;
// the fixed shape it replaced (256 threads, the whole march) took 1.37 (forward) and 1.24 (backward)
// times as long on average, 2.7 times on 64 channels of 32^3 (115 / 117 / 81 -> 42 / 50 / 34 us).
// FMA kernels (float32, odd widths): the fixed 256 and 512 threads, cut into segments until 4096 and 2048
// wavefronts were there, left rounds of workgroups part empty: 64 channels of 45x53x77 in bf16 455 / 285 ->
// 320 / 207 us (the two passes of the backward), 32 of 96^3 in float32 905 / 562 -> 602 / 418.  `alone` and
// `overlap` are fitted to those and the shapes of alone = 1, overlap = 0 on 136 problems (6 to 140 planes, 8 to 512
// channels, batches of 1 to 4; the ratio of the two predicted within 9 % in the mean, 18 % before), since with
// those one wavefront a SIMD that marched the whole way looked too cheap: 512 channels of 14x22x17 100 -> 133 us
// forward, 4 x 128 of 21x15x23 164 -> 201.  On the 136 problems the choice takes 0.92 (forward) and 0.90 (with the
// backward) of the fixed shapes' time, 1.05 at worst; with alone = 1, overlap = 0 it was 0.95 and 0.92, 1.33 at worst.
struct CostModel {
    int waves_per_simd;
    double alone, overlap;
    bool mixed;
};
static const CostModel kCostDot2F = {4, 1.0, 0.0, true}, kCostDot2B = {2, 1.0, 0.0, false};
static const CostModel kCostFmaF = {3, 2.0, 0.75, false}, kCostFmaB = {2, 3.0, 0.5, false};

static inline double launch_cost(const Tile &t, const March &m, long long nbc, int lds_floats, const CostModel &c)
{
    const int w = t.NT / 64;
    int R = kMaxLdsBytes / (lds_floats * 4);
    if (R > c.waves_per_simd * 4 / w) R = c.waves_per_simd * 4 / w;
    if (R < 1) R = 1;
    const double share = (double)(nbc * t.ntile * t.nseg) / 256.0, per = w > 3 ? (w + 3) / 4 : w / 4.0;
    auto batch = [&](int q) { return q * per + c.alone; };
    const long long ci = (nbc * t.ntile * t.nseg + 255) / 256;
    const long long full = ci / R;
    const int rem = (int)(ci - full * R);
    double T = full * batch(R);
    if (rem) T += full ? (1.0 - c.overlap) * batch(rem) + c.overlap * batch(R) * rem / R : batch(rem);
    if (c.mixed && full >= 2) T = share * batch(R) / R + 0.5 * batch(R) / R;
    const int planes = (t.SEG < m.D ? t.SEG : m.D) + (t.nseg > 1 ? 3 : 1);
    return planes * (1.0 + 0.4 / t.S) * T;
}

// The row bands (workgroups of about `targets[i]` threads of RH x RW outputs) and march segments (an
// even number of planes, `min_planes` at least) with the smallest cost.  K: the kernel whose LDS need counts.
template <class K, int N>
static inline bool cost_tile(const March &m, int RH, int RW, long long nbc, const int (&targets)[N], int min_strips,
                             int min_planes, const CostModel &model, Tile &best)
{
    double least = 0.0;
    bool found = false;
    for (int target : targets) {
        Tile t;
        if (!make_tile(m, RH, RW, target, t, min_strips)) continue;
        const int lds = K::lds_floats(t);
        if (lds * 4 > kMaxLdsBytes) continue;
        int last = 0;
        for (int n = 1; n <= 32; ++n) {
            if (n > 1 && m.D < min_planes * n) break;
            t.SEG = n == 1 ? m.D : round_up((m.D + n - 1) / n, 2);
            if (t.SEG == last) continue;
            last = t.SEG;
            t.nseg = (m.D + t.SEG - 1) / t.SEG;
            const double cost = launch_cost(t, m, nbc, lds, model);
            if (!found || cost < least) {
                found = true;
                least = cost;
                best = t;
            }
        }
    }
    return found;
}

// Column pairs of rows of any length and alignment, where they are ahead of one column a thread.
// 3-D: where the cost of their launch says so.  The times of 200 problems (3 to 255 columns, 1 to 1024 channels, 0.1 to 10 M
// voxels) follow the ratio of the two costs.  Forward, 2 x 2 outputs a thread against 4 x 1: pairs in workgroups of up to three
// wavefronts are ahead up to 0.978 of the cost (of 56 problems between 0.93 and that 0.96 of the time, the most behind 1.02),
// in larger ones, whose threads take 1.02 to 1.09 times as long, up to 0.93; workgroups of three wavefronts count 1.12
// times.  us, one column -> pairs, float32 / bf16, with that ratio: 192 channels of 23 x 29 x 33 161 -> 99 / 162 -> 99, 0.60; 32
// of 55 x 61 x 129 559 -> 371 / 563 -> 364, 0.79; 32 of 91 x 101 x 87 643 -> 585 / 661 -> 582, 0.85; 256 of 32 x 31 x 39
// 226 -> 210, 0.94; 768 of 21 x 24 x 25 279 -> 261, 0.97; 64 of 45 x 53 x 77 299 -> 300 / 306 -> 319, 0.94 with four
// wavefronts; 1024 of 6 x 3 x 7 44 -> 94 / 42 -> 95, 1.00; 16 of 106 x 82 x 73 245 -> 255 / 245 -> 274, 1.06.  Backward, 2 x 2
// outputs against 2 x 1: 1.4 (few wavefronts) to 2 times (many), so below 0.549 (1 of 143 x 135 x 135 167 -> 155 / 166 -> 143,
// 0.49; 64 of 45 x 53 x 77 547 -> 541 / 526 -> 498, 0.52; 256 of 32 x 31 x 39 493 -> 438, 0.545; 32 of 63 x 71 x 81
// 522 -> 543, 0.550; 1 of 160 x 90 x 159 134 -> 149 / 132 -> 137, 0.65; 8 of 22 x 19 x 41 62 -> 86 / 61 -> 84, 0.94).
// Not tried below 32 columns; past 192 of them pairs leave the backward one workgroup a CU (64 of 30 x 41 x 255 857 -> 1073 /
// 782 -> 949).
// 2-D: where they halve the wavefronts across a row, from 193 columns on (two for four; 161 columns, two for three, forward
// 5x5 of 256 channels of 119 x 161 110 -> 129 / 110 -> 130), and leave enough of them.  Forward up to 256 columns, 5x5 from 4 M
// pixels on (256 of 213 x 201 244 -> 215 / 244 -> 217, 32 of 226 x 241 50 -> 57 / 50 -> 59; of 281 x 281 351 -> 351).  Backward
// up to 512, from 2 M pixels on (3x3: 64 of 442 x 383 357 -> 339 / 357 -> 282, 8 of 378 x 499 53 -> 60 / 53 -> 52; 5x5: 64 of
// 151 x 223 114 -> 105 / 114 -> 98, 32 of 184 x 201 81 -> 85 / 81 -> 83); of 5x5 rows of 257 to 384 columns, where one column a
// thread takes five or six wavefronts, any (16 of 226 x 271 132 -> 94 / 132 -> 89), wider ones where segments of eight rows make
// 2048 wavefronts of four a row (16 of 270 x 401 184 -> 105 / 184 -> 98, 8 of 378 x 499 85 -> 105 / 85 -> 99).  Not where
// their segments end in a round that is nearly empty: rounds over segments below 0.6 (3x3: 0.9) of the single columns' (5x5,
// 256 of 207 x 199, 1/4 and 1/2: 476 -> 390 / 470 -> 367, 512 914 -> 730 / 897 -> 686, but 384, 2/3 and 1: 582 -> 701 /
// 576 -> 656; 3x3, 384 of 200 x 271, 1 and 1: 617 -> 642 / 413 -> 471).
// (Rows that one column a thread cannot take stay outside.)
// (true in a host build whose tests send every row they can down these kernels)
#ifndef NDC_LOOSE_EVERYWHERE
#define NDC_LOOSE_EVERYWHERE false
#endif
static inline LoosePairs loose_pairs(const KGeom &q, const March &m)
{
    const long long nbc = (long long)q.B * q.G;
    const Tuning tn = tuning();
    if (m.H == 1) {
        const long long pixels = nbc * m.D * m.W;
        LoosePairs l = {m.W > 192 && m.W <= 256 && (m.KW == 3 || pixels >= 4000 * 1000), m.W > 192 && m.W <= 512};
        if (m.KW == 3 || m.W <= 256) l.backward = l.backward && pixels >= 2000 * 1000;
        else if (m.W > 384) l.backward = l.backward && nbc * 4 * (m.D / 8) >= 2048;
        if (m.KW == 3 || m.W <= 256) {
            // rounds of the wavefronts that are resident, a segment of the march each
            auto rounds = [&](int RW) {
                Tile t;
                if (!make_tile(m, 1, RW, tn.threads_b, t)) return 0.0;
                split_march(m, nbc * t.ntile, t, kSplitWavesB);
                return (double)((nbc * t.ntile * t.nseg * (t.NT / 64) + kSplitWavesB - 1) / kSplitWavesB) / t.nseg;
            };
            const double single = rounds(1);
            l.backward = l.backward && (single == 0.0 || rounds(-2) < (m.KW == 3 ? 0.9 : 0.6) * single);
        }
        if (NDC_LOOSE_EVERYWHERE) l = {m.W >= 128 && m.W <= 256, m.W >= 128 && m.W <= 512};
        return l;
    }
    LoosePairs l = {m.W >= 2 && m.W <= 256, m.W >= 32 && m.W <= 192};
    if (NDC_LOOSE_EVERYWHERE || tn.rwf || tn.rwb || m.KH != 3 || m.KW != 3) return l;
    // the cost of pairs as a share of that of single columns (0 where those do not fit, 2 where pairs do not)
    auto ratio = [&](auto single, auto pair, int RH, const auto &targets, const CostModel &model, Tile &a, Tile &b) {
        typedef decltype(single) S;
        typedef decltype(pair) P;
        if (!cost_tile<S>(m, RH, 1, nbc, targets, 0, 4, model, a)) return 0.0;
        if (!cost_tile<P>(m, 2, -2, nbc, targets, 0, 4, model, b)) return 2.0;
        return launch_cost(b, m, nbc, P::lds_floats(b), model) / launch_cost(a, m, nbc, S::lds_floats(a), model);
    };
    const int targets_f[4] = {64, 128, tn.threads_f, 512}, targets_b[3] = {128, 256, tn.threads_b};
    Tile a, b;
    if (l.forward) {
        double r = ratio(FwdKernel<3, 3, 3, 4, 4, 1, float>(), FwdKernel<3, 3, 3, 4, 2, -2, float>(), 4, targets_f, kCostFmaF, a, b);
        if (r > 0 && r < 2) r *= (b.NT == 192 ? 1.12 : 1.0) / (a.NT == 192 ? 1.12 : 1.0);
        l.forward = r < (r > 0 && b.NT <= 192 ? 0.978 : 0.93);
    }
    if (l.backward)
        l.backward = ratio(Bwd1Kernel<3, 3, 3, 4, 2, 1, float>(), Bwd1Kernel<3, 3, 3, 4, 2, -2, float>(), 2, targets_b, kCostFmaB, a, b) < 0.549;
    return l;
}

template <int KD, int KH, int KW, int SC, int RHF, int RWF, int RHB, int RWB>
static inline void plan_lds(Plan &pl, long long nbc)
{
    if constexpr (KD == 3 && KH == 3) {
        // (153 registers a thread and more forward, 179 and more backward)
        const Tuning tn = tuning();
        const int targets_f[4] = {64, 128, tn.threads_f, 512}, targets_b[3] = {128, 256, tn.threads_b};
        if (tn.split) {
            cost_tile<FwdKernel<KD, KH, KW, SC, RHF, RWF, float>>(pl.m, RHF, RWF, nbc, targets_f, 0, 4, kCostFmaF, pl.tf);
            cost_tile<Bwd1Kernel<KD, KH, KW, SC, RHB, RWB, float>>(pl.m, RHB, RWB, nbc, targets_b, 0, 4, kCostFmaB, pl.tb);
        }
    }
    pl.lds_f = FwdKernel<KD, KH, KW, SC, RHF, RWF, float>::lds_floats(pl.tf);
    pl.lds_b1 = Bwd1Kernel<KD, KH, KW, SC, RHB, RWB, float>::lds_floats(pl.tb);
    pl.lds_b2 = Bwd2Kernel<KD, KH, KW, SC, RHB, RWB, float>::lds_floats(pl.tb);
}

static const int kDot2RH = 2;   // rows per thread of the bf16 dot2 kernels (columns: 2)

static inline bool make_plan_for(const KGeom &q, Plan &pl, int pairs, int dtype, bool matrix)
{
    pl.m = march_of(q);
    pl.dot2 = false;
    pl.mfma1 = pl.mfma2 = pl.mfmaf = false;
    // 32-bit offsets inside one (sample, channel) volume
    if ((long long)q.sc * q.SP >= (1LL << 31)) return false;
    // (aligned tensors of an even width have their own pairs)
    const bool ask = pairs >= kLooseForward && (pairs < kPairs || pl.m.W % 2);
    const LoosePairs loose = ask ? loose_pairs(q, pl.m) : LoosePairs{false, false};
    if (!find_variant(q, pl.m, pairs, loose, pl.v)) return false;
    const Tuning tn = tuning();
    if (!make_tile(pl.m, pl.v.RHF, pl.v.RWF, tn.threads_f, pl.tf)) return false;
    if (!make_tile(pl.m, pl.v.RHB, pl.v.RWB, tn.threads_b, pl.tb)) return false;
    if (tn.split && pl.m.KH == 1) {
        // 2-D: the forward keeps four wavefronts per SIMD resident, the backward kernels two
        split_march(pl.m, (long long)q.B * q.G * pl.tf.ntile, pl.tf, kSplitWavesF);
        split_march(pl.m, (long long)q.B * q.G * pl.tb.ntile, pl.tb, kSplitWavesB);
    }
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                        \
    if (NDC_IS_VARIANT(pl, kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_))                      \
        plan_lds<kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_>(pl, (long long)q.B * q.G);
    NDC_FUSED_VARIANTS(X)
#undef X
    // (their buffer addressing wants every (sample, channel group) slice below 2^31 bytes)
    if (dtype == NDC_BF16 && pairs == kPairs && pl.m.W % 2 == 0 && q.sc == 4 && pl.m.KD == 3 &&
        (long long)q.sc * q.SP * 2 < (1LL << 31) &&
        pl.m.KH == 3 && pl.m.KW == 3 && tn.dot2) {
        Tile tf, tb;
        const long long nbc = (long long)q.B * q.G;
        const int targets_f[2] = {tn.threads_f2, tn.threads_f2_wide}, targets_b[2] = {tn.threads_b2_narrow, tn.threads_b2};
        // (the matrix-instruction kernels march over whole volumes in one shape)
        const bool whole = matrix && (FwdKernelM<kDot2RH>::covers(pl.m.W) || Bwd1KernelM<kDot2RH>::covers(pl.m.W) ||
                                      Bwd2KernelM<kDot2RH>::covers(pl.m.W));
        const bool fits = whole ? make_tile(pl.m, kDot2RH, 2, tn.threads_f2, tf, FwdKernelB<kDot2RH>::kMinStrips) &&
                                      make_tile(pl.m, kDot2RH, 2, tn.threads_b2, tb)
                                : cost_tile<FwdKernelB<kDot2RH>>(pl.m, kDot2RH, 2, nbc, targets_f,
                                                                 FwdKernelB<kDot2RH>::kMinStrips, 6, kCostDot2F, tf) &&
                                      cost_tile<Bwd1KernelB<kDot2RH, true>>(pl.m, kDot2RH, 2, nbc, targets_b, 0, 6, kCostDot2B, tb);
        if (fits) {
            const int lf = FwdKernelB<kDot2RH>::lds_floats(tf);
            const int l1 = Bwd1KernelB<kDot2RH>::lds_floats(tb);
            const int l2 = Bwd2KernelB<kDot2RH>::lds_floats(tb);
            const int cap2 = kMaxLdsBytes / 4;
            if (lf <= cap2 && l1 <= cap2 && l2 <= cap2) {
                pl.dot2 = true;
                pl.tf = tf;
                pl.tb = tb;
                pl.lds_f = lf;
                pl.lds_b1 = l1;
                pl.lds_b2 = l2;
                // (pass 1 only where two of its workgroups fit a CU: with 128 columns its LDS
                // need leaves room for one, and the dot2 kernel is faster, 2.73 against 2.96 ms
                // at 64 channels of 128^3)
                pl.mfma1 = tn.mfma && matrix && Bwd1KernelM<kDot2RH>::covers(pl.m.W) &&
                           Bwd1KernelM<kDot2RH>::lds_floats(tb) <= cap2 / 2;
                pl.mfmaf = tn.mfma && matrix && FwdKernelM<kDot2RH>::covers(pl.m.W) &&
                           FwdKernelM<kDot2RH>::lds_floats(tf) <= cap2;
                pl.mfma2 = tn.mfma && matrix && Bwd2KernelM<kDot2RH>::covers(pl.m.W) &&
                           Bwd2KernelM<kDot2RH>::lds_floats(tb) <= cap2;
            }
        }
    }
    const int cap = kMaxLdsBytes / 4;
    if (pl.lds_f > cap || pl.lds_b1 > cap || pl.lds_b2 > cap) return false;
    const long long nbc = (long long)q.B * q.G;
    const long long nf = nbc * pl.tf.ntile * pl.tf.nseg, nb = nbc * pl.tb.ntile * pl.tb.nseg;
    if (nf > 0x7fffffffLL || nb > 0x7fffffffLL) return false;
    pl.nblk_f = (int)nf;
    pl.nblk_b = (int)nb;
    pl.small_f = pl.small_b = false;
    pl.nblk_f2 = pl.nblk_b2 = 0;
    if (NDC_TILES_2D && q.sc == 4 && make_tile_2d(pl.m, nbc, pl.t2)) {
        const long long image = (long long)pl.m.D * pl.m.W, pixels = nbc * image;
        const long long covered = nbc * pl.t2.ntile * pl.t2.P * pl.t2.TH;
        // (a lane takes two columns from 128 on where the width is even; whether the call's pointers allow that
        // does not count, so that every plan of a geometry agrees)
        const long long lanes = nbc * pl.m.D * round_up(pl.m.W < 128 || pl.m.W % 2 ? pl.m.W : pl.m.W / 2, 64);
        pl.small_f = pixels <= kPixelsF || (image <= 64 * 64 && pixels <= kSmallImagesF);
        pl.small_b = pixels <= kPixelsB || (image <= 32 * 32 && pixels <= kSmallImagesB);
        if (pl.m.KW == 3) {
            pl.small_f = pl.small_f && (covered <= kCovered3F || 100 * covered <= 72 * lanes);
            pl.small_b = pl.small_b && (covered <= kCovered3B || 100 * covered <= 60 * lanes);
        } else {
            pl.small_f = pl.small_f && covered <= kCoveredF;
        }
        pl.t2.PL = pairs == kPairs && pl.m.W % 2 == 0;   // pixels go in and out by pairs
        if (pl.small_f) pl.nblk_f2 = (int)(nbc * pl.t2.ntile);
        if (pl.small_b) pl.nblk_b2 = (int)(nbc * ((pl.t2.ntile + pl.t2.SEG - 1) / pl.t2.SEG));
    }
    return true;
}

// The column-pair variants hold more of a row per workgroup: where their LDS need exceeds a
// workgroup's share (wide rows of a tall image) the one-column variants may still fit, and
// those are what supported() answers for.
// matrix: the call runs the matrix-instruction family where it covers the geometry (its launch shapes
// are its own, the filter's table is the same, and workspace sizes serve both)
// pairs_ok: every activation pointer of the call is aligned to two elements
static inline bool make_plan_fresh(const KGeom &q, Plan &pl, bool pairs_ok, int dtype, bool matrix)
{
    for (int pairs = pairs_ok ? kPairs : kLoosePairs; pairs >= kSingles; --pairs)
        if (make_plan_for(q, pl, pairs, dtype, matrix)) return true;
    return false;
}

// A plan is a function of sizes, and a forward and a backward ask for it some ten times (what is
// supported, workspace sizes, the launches); the search for a launch shape takes 1-5 us.  Each thread
// keeps the plans of the last sizes it saw: an update of 64 channels of 32^3 plans for 2 us in all
// instead of 25, which a small layer waits for.
static inline bool make_plan(const KGeom &q, Plan &pl, bool pairs_ok = true, int dtype = NDC_F32, bool matrix = false)
{
#ifdef NDC_TUNING
    return make_plan_fresh(q, pl, pairs_ok, dtype, matrix);
#else
    static const int kWords = 11, kEntries = 64;
    const int key[kWords] = {q.B,  q.G,  q.m,  q.sc, q.D, q.H,
                             q.W, q.kD, q.kH, q.kW, NDC_TILES_2D * 8 + pairs_ok * 4 + matrix * 2 + (dtype == NDC_BF16)};
    struct Entry {
        int key[kWords];   // zeros where nothing is kept (a geometry has B >= 1)
        bool ok;
        Plan pl;
    };
    static thread_local Entry kept[kEntries] = {};
    unsigned at = 0;
    for (int k : key) at = at * 31 + (unsigned)k;
    Entry &e = kept[(at ^ at >> 15) % kEntries];
    if (memcmp(e.key, key, sizeof(key)) != 0) {
        e.key[0] = 0;
        e.ok = make_plan_fresh(q, e.pl, pairs_ok, dtype, matrix);
        memcpy(e.key, key, sizeof(key));
    }
    pl = e.pl;
    return e.ok;
#endif
}

static inline bool supported(const KGeom &q)
{
    Plan pl;
    return make_plan(q, pl, false);
}

template <typename T> static inline bool pair_aligned(const void *p)
{
    return p == nullptr || ((uintptr_t)p % (2 * sizeof(T))) == 0;
}

static inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// scratch: gt1 (activation dtype) | pass-1 partials | pass-2 partials
static inline size_t backward_ws(const KGeom &q, int dtype, int /*need_gh*/, int /*need_gb*/)
{
    // sized for whichever variant the call ends up with (aligned pairs or not)
    Plan a, b;
    if (!make_plan(q, a, false, dtype)) return 0;
    const bool has_b = make_plan(q, b, true, dtype);
    size_t nblk = has_b && b.nblk_b > a.nblk_b ? b.nblk_b : a.nblk_b;
    // ... and whichever kernel family
    Plan mx;
    if (make_plan(q, mx, true, dtype, true) && (size_t)mx.nblk_b > nblk) nblk = mx.nblk_b;
    const size_t esz = dtype == NDC_BF16 ? 2 : 4;
    const size_t n_x = (size_t)q.B * q.G * q.SP;
    const size_t kt = (size_t)q.sc * q.KT;
    const size_t tabs = has_b && b.dot2 ? align256((size_t)q.G * kTabWords * 4) : 0;
    const size_t march = align256(n_x * esz) + align256(nblk * kt * 4) + align256(nblk * (kt + q.sc) * 4) + tabs;
    const size_t tiles = align256((size_t)a.nblk_b2 * (kt + q.sc) * 4);
    return march > tiles ? march : tiles;
}

// bytes of scratch the forward call needs (the packed tap tables of the bf16 dot2 kernels)
static inline size_t forward_ws(const KGeom &q, int dtype)
{
    Plan pl;
    if (!make_plan(q, pl, true, dtype) || !pl.dot2) return 0;
    return align256((size_t)q.G * kTabWords * 4);
}

// whether backward() reads the forward's s/d and n/d for this geometry: every fused kernel
// family has that form
static inline bool backward_uses_saved(const KGeom &q, int dtype)
{
    Plan pl;
    return make_plan(q, pl, true, dtype);
}

template <class BE, typename T> struct Dot2Launch {
    static int fwd(const FwdParams<T> &, const Plan &, void *) { return NDC_ERR_GEOMETRY; }
    static int bwd1(const BwdParams<T> &, const Plan &, void *, bool) { return NDC_ERR_GEOMETRY; }
    static int bwd2(const BwdParams<T> &, const Plan &, void *, bool) { return NDC_ERR_GEOMETRY; }
};
template <class BE> struct Dot2Launch<BE, bf16_t> {
    template <bool NT> static int fwd_dot2(const FwdParams<bf16_t> &p, const Plan &pl, void *stream)
    {
        if (p.s_over_den && p.ratio)
            return BE::template block_kernel<FwdKernelB<kDot2RH, true, NT>>(p, pl.nblk_f, pl.tf.NT, pl.lds_f, stream);
        return BE::template block_kernel<FwdKernelB<kDot2RH, false, NT>>(p, pl.nblk_f, pl.tf.NT, pl.lds_f, stream);
    }
    template <bool NT> static int bwd1_dot2(const BwdParams<bf16_t> &p, const Plan &pl, void *stream, bool saved)
    {
        typedef Bwd1KernelB<kDot2RH, true, NT> KS;
        if (saved) return BE::template block_kernel<KS>(p, pl.nblk_b, pl.tb.NT, KS::lds_floats(pl.tb), stream);
        return BE::template block_kernel<Bwd1KernelB<kDot2RH, false, NT>>(p, pl.nblk_b, pl.tb.NT, pl.lds_b1, stream);
    }
    template <bool NT> static int bwd2_dot2(const BwdParams<bf16_t> &p, const Plan &pl, void *stream, bool saved)
    {
        typedef Bwd2KernelB<kDot2RH, true, NT> KS;
        if (saved) return BE::template block_kernel<KS>(p, pl.nblk_b, pl.tb.NT, KS::lds_floats(pl.tb), stream);
        return BE::template block_kernel<Bwd2KernelB<kDot2RH, false, NT>>(p, pl.nblk_b, pl.tb.NT, pl.lds_b2, stream);
    }
    // (rows of whole 128-byte lines: see FwdKernelB)
    static bool whole_lines(const Plan &pl) { return pl.m.W % 64 == 0; }

    static int fwd(const FwdParams<bf16_t> &p, const Plan &pl, void *stream)
    {
        if (pl.mfmaf)
            return BE::template block_kernel<FwdKernelM<kDot2RH>>(p, pl.nblk_f, pl.tf.NT,
                                                                   FwdKernelM<kDot2RH>::lds_floats(pl.tf), stream);
        return whole_lines(pl) ? fwd_dot2<true>(p, pl, stream) : fwd_dot2<false>(p, pl, stream);
    }
    // saved: the call brought the forward's s/d and n/d
    static int bwd1(const BwdParams<bf16_t> &p, const Plan &pl, void *stream, bool saved)
    {
        if (saved && pl.mfma1)
            return BE::template block_kernel<Bwd1KernelM<kDot2RH>>(
                p, pl.nblk_b, pl.tb.NT, Bwd1KernelM<kDot2RH>::lds_floats(pl.tb), stream);
        return whole_lines(pl) ? bwd1_dot2<true>(p, pl, stream, saved) : bwd1_dot2<false>(p, pl, stream, saved);
    }
    static int bwd2(const BwdParams<bf16_t> &p, const Plan &pl, void *stream, bool saved)
    {
        if (saved && pl.mfma2)
            return BE::template block_kernel<Bwd2KernelM<kDot2RH>>(
                p, pl.nblk_b, pl.tb.NT, Bwd2KernelM<kDot2RH>::lds_floats(pl.tb), stream);
        return whole_lines(pl) ? bwd2_dot2<true>(p, pl, stream, saved) : bwd2_dot2<false>(p, pl, stream, saved);
    }
};

// the packed filter tables of the bf16 dot2 kernels: G * kTabWords words from h
template <class BE> static int prepare_taps(const KGeom &q, const float *h, float *tab, void *stream)
{
    return BE::elementwise((long long)q.G * kTabWords, stream,
                           [=] NDC_LAMBDA(long long idx) { prep_tables(idx, h, tab); });
}

// h = max(h0, 0) and the tables of h, in one launch: a filter of 4 x 27 taps has fewer values than its table words
template <class BE> static int rectify_and_prepare(const KGeom &q, const float *h0, float *h, float *tab, void *stream)
{
    return BE::elementwise((long long)q.G * kTabWords, stream, [=] NDC_LAMBDA(long long idx) {
        const long long c = idx / kTabWords, e = idx % kTabWords;
        if (e < 4 * 27) h[c * 4 * 27 + e] = floor_f(h0[c * 4 * 27 + e], 0.f);
        prep_tables(idx, Rectified{h0}, tab);
    });
}

// f(kernel type tag): the instance of a one-shot 2-D kernel for this plan
template <template <int, int, typename> class Kernel, typename T, class F> static int with_tile_2d(const Plan &pl, F f)
{
    if (pl.m.KD == 5) return pl.t2.P == 16 ? f((Kernel<5, 16, T> *)nullptr) : f((Kernel<5, 32, T> *)nullptr);
    return pl.t2.P == 16 ? f((Kernel<3, 16, T> *)nullptr) : f((Kernel<3, 32, T> *)nullptr);
}

template <class BE, typename T>
int forward(const KGeom &q, const T *x, const T *z, const float *h, const float *bias,
                   T *out, T *t1, T *s_over_den, T *ratio, const float *taps, void *ws,
                   void *stream)
{
    // taps: packed filter tables prepared earlier for this h (prepare_taps), or null: then
    // they are packed into ws by a small launch ahead of the kernel
    Plan pl;
    const bool pairs = pair_aligned<T>(x) && pair_aligned<T>(z) && pair_aligned<T>(out) &&
                       pair_aligned<T>(t1) && pair_aligned<T>(s_over_den) && pair_aligned<T>(ratio);
    const int dtype = sizeof(T) == 2 ? NDC_BF16 : NDC_F32;
    if (!make_plan(q, pl, pairs, (ws || taps) ? dtype : NDC_F32, q.matrix != 0)) return NDC_ERR_GEOMETRY;
    FwdParams<T> p;
    p.wtab = nullptr;
    p.x = x;
    p.z = z;
    p.h = h;
    p.bias = bias;
    p.out = out;
    p.t1 = t1;
    p.s_over_den = s_over_den;
    p.ratio = ratio;
    p.B = q.B;
    p.C = q.G;
    p.D = pl.m.D;
    p.H = pl.m.H;
    p.W = pl.m.W;
    p.relu = q.relu;
    p.eps = q.eps;
    p.t = pl.tf;
    if (pl.dot2) {
        if (taps) {
            p.wtab = taps;
        } else {
            float *tab = (float *)ws;
            const int st = prepare_taps<BE>(q, h, tab, stream);
            if (st) return st;
            p.wtab = tab;
        }
        return Dot2Launch<BE, T>::fwd(p, pl, stream);
    }
    if (pl.small_f) {
        p.t = pl.t2;
        return with_tile_2d<Fwd2D, T>(pl, [&](auto *tag) {
            typedef std::remove_pointer_t<decltype(tag)> KS;
            return BE::template block_kernel<KS>(p, pl.nblk_f2, pl.t2.NT, KS::lds_floats(pl.t2), stream);
        });
    }
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                          \
    if (NDC_IS_VARIANT(pl, kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_))                        \
        return BE::template block_kernel<FwdKernel<kd_, kh_, kw_, sc_, rhf_, rwf_, T>>(        \
            p, pl.nblk_f, pl.tf.NT, pl.lds_f, stream);
    NDC_FUSED_VARIANTS(X)
#undef X
    return NDC_ERR_GEOMETRY;
}

template <class BE, typename T>
int backward(const KGeom &q, const T *x, const T *z, const T *t1, const T *s_over_den,
                    const T *ratio, const float *h, const float *bias, const T *gout, T *gx,
                    T *gz, float *gh, float *gb, const float *taps, void *ws, void *stream,
                    float *pass_ms = nullptr)
{
    // pass_ms (optional, 3 floats): device time of pass 1, pass 2 and the partial-sum
    // reduction, taken with events on `stream`; makes the call synchronous
    typename BE::Timer tm(pass_ms != nullptr, stream);
    Plan pl;
    const bool pairs = pair_aligned<T>(x) && pair_aligned<T>(z) && pair_aligned<T>(t1) &&
                       pair_aligned<T>(gout) && pair_aligned<T>(gx) && pair_aligned<T>(gz) &&
                       pair_aligned<T>(s_over_den) && pair_aligned<T>(ratio);
    const bool saved = s_over_den != nullptr && ratio != nullptr;
    const int dtype = sizeof(T) == 2 ? NDC_BF16 : NDC_F32;
    if (!make_plan(q, pl, pairs, dtype, q.matrix != 0)) return NDC_ERR_GEOMETRY;
    const size_t n_x = (size_t)q.B * q.G * q.SP;
    const int kt = q.sc * q.KT;
    char *w = (char *)ws;
    T *gt1 = (T *)w;
    w += align256(n_x * sizeof(T));
    float *part1 = (float *)w;
    w += align256((size_t)pl.nblk_b * kt * 4);
    float *part2 = (float *)w;
    w += align256((size_t)pl.nblk_b * (kt + q.sc) * 4);
    float *tab = (float *)w;

    BwdParams<T> p;
    p.x = x;
    p.z = z;
    p.t1 = t1;
    p.gout = gout;
    p.s_over_den = s_over_den;
    p.ratio = ratio;
    p.h = h;
    p.bias = bias;
    p.gx = gx;
    p.gz = gz;
    p.gt1 = gt1;
    p.wtab = nullptr;
    p.need_gh = gh != nullptr;
    p.need_gb = gb != nullptr;
    p.B = q.B;
    p.C = q.G;
    p.D = pl.m.D;
    p.H = pl.m.H;
    p.W = pl.m.W;
    p.relu = q.relu;
    p.eps = q.eps;
    p.t = pl.tb;

    int st = NDC_ERR_GEOMETRY;
    const int C = q.G, SC = q.sc, B = q.B;
    // (gh and gb in one launch: outputs [0, C kt) are gh, the C SC after them gb)
    const int n_gh = gh ? C * kt : 0, n_gb = gb ? C * SC : 0, gate = q.gate;
    auto put = [=] NDC_LAMBDA(int o, float v) {
        if (o < n_gh) gh[o] = gate && h[o] <= 0.f ? 0.f : v; else gb[o - n_gh] = v;
    };
    if (pl.small_b && saved) {
        float *part = (float *)ws;
        p.t = pl.t2;
        p.part = part;
        p.part_stride = kt + SC;
        st = with_tile_2d<Bwd2D, T>(pl, [&](auto *tag) {
            typedef std::remove_pointer_t<decltype(tag)> KS;
            return BE::template block_kernel<KS>(p, pl.nblk_b2, pl.t2.NT, KS::lds_floats(pl.t2), stream);
        });
        if (st) return st;
        tm.mark();
        tm.mark();
        if (n_gh + n_gb) {
            const int ntile = (pl.t2.ntile + pl.t2.SEG - 1) / pl.t2.SEG;
            st = BE::strided_sum(n_gh + n_gb, B * ntile, stream, put, [=] NDC_LAMBDA(int o, int pi) {
                const int c = o < n_gh ? o / kt : (o - n_gh) / SC, r = o < n_gh ? o % kt : kt + (o - n_gh) % SC;
                return part[(((long long)(pi / ntile) * C + c) * ntile + pi % ntile) * (kt + SC) + r];
            });
            if (st) return st;
        }
        tm.mark();
        tm.finish(pass_ms, 3);
        return NDC_OK;
    }
    p.part = part1;
    p.part_stride = kt;
    if (pl.dot2) {
        if (taps) {
            p.wtab = taps;
        } else {
            st = prepare_taps<BE>(q, h, tab, stream);
            if (st) return st;
            p.wtab = tab;
        }
        st = Dot2Launch<BE, T>::bwd1(p, pl, stream, saved);
    } else {
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                          \
    if (NDC_IS_VARIANT(pl, kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)) {                      \
        if (saved)                                                                             \
            st = BE::template block_kernel<Bwd1Kernel<kd_, kh_, kw_, sc_, rhb_, rwb_, T, true>>(\
                p, pl.nblk_b, pl.tb.NT, pl.lds_b1, stream);                                    \
        else                                                                                   \
            st = BE::template block_kernel<Bwd1Kernel<kd_, kh_, kw_, sc_, rhb_, rwb_, T>>(     \
                p, pl.nblk_b, pl.tb.NT, pl.lds_b1, stream);                                    \
    }
        NDC_FUSED_VARIANTS(X)
#undef X
    }
    if (st) return st;
    tm.mark();
    if (!gz && !gh && !gb) {
        tm.finish(pass_ms, 3);
        return NDC_OK;
    }

    p.part = part2;
    p.part_stride = kt + q.sc;
    st = NDC_ERR_GEOMETRY;
    if (pl.dot2) {
        st = Dot2Launch<BE, T>::bwd2(p, pl, stream, saved);
    } else {
#define X(kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)                                          \
    if (NDC_IS_VARIANT(pl, kd_, kh_, kw_, sc_, rhf_, rwf_, rhb_, rwb_)) {                      \
        typedef Bwd2Kernel<kd_, kh_, kw_, sc_, rhb_, rwb_, T, true> KS;                        \
        if (saved)                                                                             \
            st = BE::template block_kernel<KS>(p, pl.nblk_b, pl.tb.NT, KS::lds_floats(pl.tb),  \
                                               stream);                                        \
        else                                                                                   \
            st = BE::template block_kernel<Bwd2Kernel<kd_, kh_, kw_, sc_, rhb_, rwb_, T>>(     \
                p, pl.nblk_b, pl.tb.NT, pl.lds_b2, stream);                                    \
    }
        NDC_FUSED_VARIANTS(X)
#undef X
    }
    if (st) return st;
    tm.mark();

    // combine the per-workgroup partial sums: a fixed association, so results are reproducible
    const int ntile = pl.tb.ntile * pl.tb.nseg;
    if (n_gh + n_gb) {
        st = BE::strided_sum(n_gh + n_gb, B * ntile, stream, put, [=] NDC_LAMBDA(int o, int pi) {
            if (o < n_gh) {
                const int c = o / kt, r = o % kt;
                const long long blk = ((long long)(pi / ntile) * C + c) * ntile + pi % ntile;
                return part1[blk * kt + r] + part2[blk * (kt + SC) + r];
            }
            const int c = (o - n_gh) / SC, i = (o - n_gh) % SC;
            const long long blk = ((long long)(pi / ntile) * C + c) * ntile + pi % ntile;
            return part2[blk * (kt + SC) + kt + i];
        });
        if (st) return st;
    }
    tm.mark();
    tm.finish(pass_ms, 3);
    return NDC_OK;
}

// the two above for one backend and storage type, to declare (`extern template`) or instantiate
#define NDC_FUSED_ENTRY_POINTS(KIND, T)                                                            \
    KIND int forward<Backend, T>(const KGeom &, const T *, const T *, const float *, const float *, \
                                 T *, T *, T *, T *, const float *, void *, void *);               \
    KIND int backward<Backend, T>(const KGeom &, const T *, const T *, const T *, const T *,        \
                                  const T *, const float *, const float *, const T *, T *, T *,     \
                                  float *, float *, const float *, void *, void *, float *);

}  // namespace fused
}  // namespace ndc
