// Which kernel serves a GEMM call (and one quantizer's): the rules, apart from the kernels and the
// launches, so that they can be asked on any machine.  A call's sizes, whether it brings a split-K
// workspace and the device's CUs decide; every rule gives both sides' measurements.
#pragma once

#include <algorithm>

#include "ckh_common.h"

namespace ckh {

constexpr int kTile = 256;       // rows and columns of the tile kernels' output tiles
constexpr int kTileSlots = 256;  // workgroups that can hold such a tile at once: one per CU
constexpr int64_t kPartialBytes = int64_t(kTile) * kTile * 4;  // one fp32 partial tile

// Activations of at most this many rows take the skinny kernels, or few-row small tiles.
constexpr int kSkinnyMaxM = 64;
// From 17 rows and this N on, MXFP8 small tiles serve them instead (mx_few_rows_tile).
constexpr int kSkinnySmallN = 8192;

struct SplitPlan {
    int S = 1;   // K ranges (1: no split)
    int ks = 0;  // 64-wide stages (MXFP8, FP8) or 256-wide groups (NVFP4) per range
    int nw = 4;  // 4: full tiles, 2: half tiles
};

struct SmallTile {
    int tm, tn;
};

// A skinny kernel's shape: waves per workgroup, 32-row weight tiles per workgroup, 32-row
// activation tiles, activation rows staged in LDS (MXFP8) or decoded to it (NVFP4; 0: each lane
// decodes its own), and rows of activation codes staged in LDS (NVFP4 only).
struct SkinnyForm {
    int waves, weight_tiles, act_tiles, act_rows, code_rows;
};

struct Route {
    enum Kind { kSkinny, kSmall, kSplit, kTiles } kind = kTiles;
    int form = 0;                             // index of the skinny form or small tile
    SplitPlan split;                          // kSplit
    int n_full = 0, n_half = 0, n_pref = 0;   // kTiles: whole tiles, tiles run as two halves, prefetch workgroups
};

// ------------------------------------------------------------------ MXFP8, per-tensor FP8
// The skinny form by activation size (N = 18432, K = 3072: M = 1 12.7 us, M = 16 15.4 us).  With
// 16 activation rows the waves per workgroup follow N: 2 waves when there are at least 256
// workgroups (M = 16, N = 18432: 14.6 against 15.4 us with 4), 8 when there are fewer than 128
// (N = 3072, K = 12288: 16.6 against 17.2 us; with 2 waves 25.9 us).  With 4-8 rows and N above
// 16384, 2 waves rather than 8 (M = 8, N = 18432, K = 3072 13.4 against 14.5 us; N = 24576 14.9
// against 15.8; M = 4 13.1 against 13.6; M = 1 and 2 and N = 16384 equal).  From 17 rows on this
// kernel serves what mx_few_rows_tile leaves: N below 8192, where its waves' split of K keeps
// more of the chip busy than small tiles would (32 x 5120 x 5120 11.6 against 16.1 us, 64 x 5120
// x 12288 27.7 against 37.0); short K; 17-32 rows of a narrow layer; and N beyond one round of 64
// x 128 tiles.  There the activation is staged through LDS too, 32 or 64 rows (N = 5120, K =
// 5120, M = 32 10.8 against 16.5 us with the fragments loaded into registers; M = 64, K = 13824
// 29.3 against 47.4), and the choice follows how many workgroups one round holds: 17-32 rows 4
// waves and two weight tiles up to N = 16384 (K = 5120 18.7 against 19.8 us with one tile); then
// one tile with 2 waves (20 x 18432 x 3072 16.4 against 17.3 with 4) or, from K = 4096 on, 4 (32
// x 18432 x 12288 57.4 against 57.7 with 2 waves and two tiles); 2 waves and two tiles beyond N =
// 24576 (20 x 32768 x 3072 20.2 against 22.0); 33-64 rows 2 waves and one tile (three workgroups
// of 48 KB per CU) up to N = 24576 (64 x 18432 x 3072 20.6 against 21.6 with two tiles), two
// tiles beyond (64 x 32768 x 3072 25.2 against 29.1).
// The NVFP4 skinny kernel's form (128-byte chunks, two in flight per wave) measured slower
// here, where a chunk costs only a few MFMAs: M = 1 14.5 against 12.9 us, M = 16 15.9 against
// 15.5, M = 64 29.6 against 26.5 (same process).
constexpr SkinnyForm kMxSkinny[] = {{8, 1, 1, 8},  {2, 1, 1, 8},  {8, 1, 1, 16}, {4, 1, 1, 16}, {2, 1, 1, 16},
                                    {8, 1, 1, 32}, {4, 2, 1, 32}, {2, 1, 1, 32}, {2, 2, 1, 32}, {4, 1, 1, 32},
                                    {4, 1, 2, 64}, {2, 2, 2, 64}, {2, 1, 2, 64}};

inline int mx_skinny_form(int M, int N, int K) {
    if (M <= 8) return M >= 4 && N > 16384 ? 1 : 0;
    if (M <= 16) return N >= 8192 ? 4 : N >= 4096 ? 3 : 2;
    if (M <= 32) return N > 24576 ? 8 : N > 16384 ? (K <= 4096 ? 7 : 9) : N >= kSkinnySmallN ? 6 : 5;
    return N < kSkinnySmallN ? 10 : N > 24576 ? 11 : 12;
}

// Split-K: a grid of at most half as many 256 x 256 tiles as CUs leaves most CUs idle
// while each tile walks all of K.  Such a grid with long K instead runs S K ranges of every
// tile (each of ks stages, a multiple of 4, at least kMinSplitStages) as S times as many
// workgroups, at most one per CU, which write fp32 partial tiles to the caller's workspace;
// a second launch adds them.  A partial tile (256 KB) costs about as much memory traffic
// to write and again to read back as 8 stages of operand loads, so short K (fewer than
// kMinSplitK stages) keeps whole-K half tiles instead.  With at most a quarter as many
// tiles as CUs the split runs 256 x 128 half tiles, at least two K ranges each: a half
// tile's stage costs ~53% of a full tile's (C4's last round) and its partial (128 KB) half
// as much traffic, so for the same workgroups the partials move half the bytes.  Half
// tiles split from kMinSplitKHalf stages on, and below kMinSplitK stages on at most
// kShortSplitSlots workgroups (same process, against whole-K half tiles: 512 x 4096 x 3072
// 23.0 against 28.5 us, 22.6 with 256 workgroups; 256 x 9216 x 3072 24.8 against 29.3;
// 256 x 3072 x 3072 17.9 against 21.2; with that cap on long K too, 256 x 5120 x 13824
// took 38.3 against 36.0 us).  Full tiles split only into three ranges or more: two
// ranges give as many workgroups as whole-K half tiles, which need no partials (same
// process: 256 x 32768 x 5120 57.6 against 66.6 us split, 384 x 12288 x 6144 54.0 against
// 56.2; with three, 256 x 18432 x 8192 60.7 split against 71.2).
// Measured, graph-timed: M = 256, N = 5120, K = 13824 40.5 us split in full tiles against
// 110.8 us whole-K half tiles; N = 13824, K = 5120 40.1 against 46.9 us; N = 18432,
// K = 3072 38.3 against 32.1 us (not split).  Half tiles against full tiles in the split
// (same process): 256 x 4096 x 4096 20.9 against 27.1 us, 256 x 5120 x 13824 36.3 against
// 40.4, 512 x 3072 x 13824 38.6 against 42.5, 256 x 13824 x 5120 38.7 against 40.6.
constexpr int kMinSplitStages = 12;
constexpr int kMinSplitK = 64;      // stages
constexpr int kMinSplitKHalf = 32;  // stages, half tiles
constexpr int kShortSplitSlots = 224;

inline SplitPlan mx_split_plan(int M, int N, int K) {
    SplitPlan sp;
    if (M <= kSkinnyMaxM) return sp;
    const int tiles = static_cast<int>(cdiv(M, kTile) * cdiv(N, kTile));
    const int KT = static_cast<int>(cdiv(K, 64));
    const bool half = tiles <= kTileSlots / 4;
    if (tiles > kTileSlots / 2 || KT < (half ? kMinSplitKHalf : kMinSplitK)) return sp;
    const int units = half ? 2 * tiles : tiles;
    const int slots = half && KT < kMinSplitK ? kShortSplitSlots : kTileSlots;
    const int S = std::min(slots / units, KT / kMinSplitStages);
    if (S < (half ? 2 : 3)) return sp;
    sp.ks = static_cast<int>(rup(cdiv(KT, S), 4));
    sp.S = static_cast<int>(cdiv(KT, sp.ks));
    sp.nw = half ? 2 : 4;
    return sp;
}

// one partial tile (or two partial half tiles) per tile and K range
inline int64_t mx_split_workspace_bytes(int M, int N, int K) {
    const SplitPlan sp = mx_split_plan(M, N, K);
    if (sp.S < 2) return 0;
    return cdiv(M, kTile) * cdiv(N, kTile) * sp.S * kPartialBytes;
}

// Small tiles (gemm_mid.h): the first of these whose grid fits the CUs in one round.  The
// order is by operand rows, i.e. by time: over 200 measured shapes the first that fits was
// within 3% of the fastest that fits.  Larger tiles than these (or a second round) were slower
// than the 256 x 256 kernel's half tiles.
constexpr SmallTile kMxSmall[] = {{64, 64}, {128, 64}, {128, 96}, {128, 128}, {128, 160}, {128, 192}, {64, 128}};
constexpr int kMxSmallWide = 6;  // 64 x 128, for at most 64 rows only (mx_small_tile looks at those before it)

// Index of the small tile to use, or -1: the estimated time (us) of the first that fits against
// that of the 256 x 256 kernel.  Fitted to the same shapes:
//   small tiles  2.0 + 0.0165 rows + 0.00228 rows per 128-byte stage (rows = TM + TN);
//   split-K      14.7 + 0.575 per stage of a K range in half tiles, 1.09 in full tiles (two
//                launches; 200 x 5120 x 13824, six ranges of 36: 35.4 measured, small tiles 50);
//   half tiles   6.2 + 0.4 per stage of K (200 x 21504 x 512: 9.5 measured, small tiles 12.1).
// With K not a multiple of 128 a stage's piece of a row lies in two cache lines, and lines are
// what a CU's intake is counted in: the terms per stage of the one-launch forms take 1.45 x (84 x
// 12624 x 9824 53.1 against 38.9, 360 x 9584 x 2400 23.6 against 17.3), 1.33 x where more than 6
// tiles share a weight row, part of which then comes from L2 (691 x 1312 x 5824 16.2 against 17.5,
// 1024 x 4368 x 13728 103 against 81 split with the weight read anew, 80 against 72 with it in the
// caches; 1.1 x chose the small tiles there).  118 x 2448 x 6304: small tiles 25.0, split-K 21.0; 460
// x 3112 x 9312 43.5 and 37.5.  Over 4,200 shapes of 65-1400 rows the small tiles it chooses take
// 0.57 of the time; 1% of the choices are more than 5% slower, at most 20%, where the two
// estimates are close.
inline int mx_small_tile(int M, int N, int K, const SplitPlan& sp, int cus) {
    for (int i = 0; i < kMxSmallWide; ++i) {
        const SmallTile t = kMxSmall[i];
        if (cdiv(M, t.tm) * cdiv(N, t.tn) > cus) continue;
        const double rows = t.tm + t.tn;
        const double lines = K % 128 == 0 ? 1.0 : cdiv(M, t.tm) <= 6 ? 1.45 : 1.33;
        const double mid = 2.0 + 0.0165 * rows + 0.00228 * rows * lines * static_cast<double>(cdiv(K, 128));
        const double big = sp.S > 1 ? 14.7 + (sp.nw == 2 ? 0.575 : 1.09) * sp.ks
                                    : 6.2 + 0.4 * lines * static_cast<double>(cdiv(K, 64));
        return mid < big ? i : -1;
    }
    return -1;
}

// The small tile for at most 64 rows, or -1 for the skinny kernel: from 17 rows and N = 8192 on,
// 64 x 64 or 64 x 128, whichever fits in one round, where K is long enough to make up for the ring's
// fill and the one workgroup per CU.  Measured against the skinny kernel on 3,600 shapes, graph-timed
// both with every call's weight read anew and with one weight that stays in the caches (small tile /
// skinny, us, anew; the same kept):
//   33-64 rows  64 x 64 at any K: 64 x 8192 x 12288 40.5 / 43.5; 25.2 / 42.8, 48 x 12288 x 3072 13.1 /
//               15.2; 10.1 / 14.1; the mean of all 0.91; 0.72.  64 x 128 from K = 1280 on (640 above N =
//               24576): 52 x 19808 x 512 7.4 / 5.9; 6.5 / 5.2, 57 x 17328 x 1024 9.6 / 8.1; 8.2 / 7.6,
//               64 x 24576 x 5120 33.6 / 37.6; 24.0 / 36.8.
//   17-32 rows  they gain only where the weight is in the caches, so they stay where they are level
//               otherwise (in the mean 1.00; 0.82 kept): 64 x 64 above N = 10240 from K = 3072 on (25 x
//               8688 x 1024 6.8 / 5.2; 5.9 / 4.2, 32 x 9688 x 2624 11.6 / 10.6; 8.4 / 6.6); 64 x 128
//               above K = 4096, up to N = 24576 only with whole lines (K a multiple of 128; 29 x 20408 x
//               6880 42.1 / 36.7; 26.7 / 35.7).
// With 16 rows they are level.
inline int mx_few_rows_tile(int M, int N, int K, int cus) {
    if (M <= 16 || N < kSkinnySmallN) return -1;
    const bool few = M <= 32;
    if (cdiv(N, 64) <= cus) return few && (N <= 10240 || K < 3072) ? -1 : 0;
    if (cdiv(N, 128) > cus) return -1;
    if (few) return K <= 4096 || (K % 128 && N <= 24576) ? -1 : kMxSmallWide;
    return K < (N <= 24576 ? 1280 : 640) ? -1 : kMxSmallWide;
}

// The 256 x 256 tiles run one per CU in rounds.  When the last round would be at most
// half full (e.g. 864 tiles = 3 rounds + 96), its tiles run as twice as many 256 x 128
// half tiles (about 55% of a full tile's time each), in the same grid.  (A grid of at most half as
// many tiles as CUs with no workspace for split-K runs all of its tiles as half tiles: 256 x 18432
// x 3072 measured 31.9 against 41.3 us.)
inline void tile_rounds(Route& r, int M, int N) {
    const int tiles = static_cast<int>(cdiv(M, kTile) * cdiv(N, kTile));
    const int tail = tiles > kTileSlots ? tiles % kTileSlots : tiles;
    r.kind = Route::kTiles;
    r.n_half = (tail > 0 && tail <= kTileSlots / 2) ? tail : 0;
    r.n_full = tiles - r.n_half;
}

// Activations of at most kSkinnyMaxM rows take the skinny kernel, a few hundred rows the small
// tiles, and small grids with long K split K when the caller gives a workspace; the rest are
// 256 x 256 tiles, a grid of one round of which fills the remaining CUs with weight-prefetch
// workgroups.
inline Route mx_route(int M, int N, int K, bool workspace, int cus) {
    Route r;
    if (M <= kSkinnyMaxM) {
        r.form = mx_few_rows_tile(M, N, K, cus);
        r.kind = r.form >= 0 ? Route::kSmall : Route::kSkinny;
        if (r.form < 0) r.form = mx_skinny_form(M, N, K);
        return r;
    }
    r.split = mx_split_plan(M, N, K);
    if (!workspace) r.split.S = 1;
    r.form = mx_small_tile(M, N, K, r.split, cus);
    if (r.form >= 0) {
        r.kind = Route::kSmall;
        return r;
    }
    r.kind = Route::kSplit;
    if (r.split.S > 1) return r;
    tile_rounds(r, M, N);
    // (the CUs the device has, which a partitioned GPU reduces: prefetch workgroups that
    // found no idle CU would run after the tiles, for nothing)
    r.n_pref = std::max(0, cus - r.n_full - 2 * r.n_half);
    return r;
}

// ------------------------------------------------------------------ NVFP4
// The skinny form by activation size; two chunks in flight per wave.  Measured (graph-timed,
// K = 5120, N = 13824): M = 1 12.5 us, M = 8 13.0 us, M = 16 16.0 us; 8 waves, 3 chunks in flight, or
// activation fragments decoded in registers were 10-20% slower at M <= 8.  With fewer than
// 256 workgroups (N < 8192) 8 waves per workgroup pay instead (same process, against 4):
// M = 16, N = 5120, K = 13824 18.8 against 22.1 us; M = 16, N = 3072, K = 12288 17.0
// against 20.0; M = 1, N = 5120, K = 5120 8.1 against 8.8 (for the staged 32-row
// activation 8 waves measured 9-11% slower).  For M > 16 two
// weight tiles per workgroup halve the activation decoding per weight byte, which pays
// while N gives enough workgroups (M = 64: N = 13824 19.4 against 24.8 us with one tile;
// N = 5120, K = 13824 27.5 against 32.4 us with two).  With one tile (N < 8192) the
// activation codes are staged in LDS by whole-line loads rather than loaded by each lane
// (M = 32, N = 5120, K = 5120 10.0 against 10.4 us; M = 64, N = 3072, K = 12288 22.3
// against 24.7; M = 64, N = 5120, K = 13824 25.1 against 26.6); with two tiles that
// measured no better (19.6 against 19.5 us at M = 64, N = 13824).
constexpr SkinnyForm kNvSkinny[] = {{4, 1, 1, 8, 0}, {8, 1, 1, 8, 0},  {4, 1, 1, 16, 0}, {8, 1, 1, 16, 0},
                                    {4, 2, 1, 0, 0}, {4, 1, 1, 0, 32}, {4, 2, 2, 0, 0},  {4, 1, 2, 0, 64}};

inline int nv_skinny_form(int M, int N) { return (M <= 8 ? 0 : M <= 16 ? 2 : M <= 32 ? 4 : 6) + (N >= 8192 ? 0 : 1); }

// Split-K: a grid of at most 128 tiles (half the CUs) with at least kNvMinSplitK groups of
// 256 elements runs S K ranges of every tile (each of ks groups, the last one fewer, at
// least kNvMinSplitGroups) as S times as many workgroups, at most 256, which write fp32
// partial tiles to the caller's workspace; a second launch adds them.  A group costs about
// 4 us of MFMA time per tile and a partial tile's round trip about as much as one group.
// Ranges of an odd number of groups end mid-pair (measured against ranges rounded up to an
// even count, same process: M = 256, N = 13824, K = 5120, four ranges of 5 instead of 6, 6,
// 6, 2: 48.7 against 53.8 us; M = 300, N = 2000, K = 4160 35.0 against 39.6; M = 2048, N =
// 4096, K = 5376 84.6 against 90.1).  Minimum range lengths of 2, 3, 6 and 8 groups
// measured no better than 4 over six shapes (2: 300 x 2000 x 4160 30.9 against 34.4 us but
// 256 x 3072 x 12288 36.5 against 35.4; 8: up to 40% slower).  Grids of at most
// kNvHalfSplitTiles tiles split their 256 x 128 column halves instead (twice the units,
// half the ranges: less partial traffic per unit of work), also in ranges of at least
// kNvMinSplitGroups (3 measured 2-4% faster on three shapes but 16% slower on 512 x 3072 x
// 3072; 2 slower on four of five).  Grids of 65-128 tiles split whole tiles only into three
// ranges or more and from kNvMinSplitKFull groups on; otherwise they run as one round of
// whole-K half tiles, which write no partials (same process, split against half tiles: two
// ranges, 256 x 32768 x 5120 86.0 against 73.8 us, 2048 x 4096 x 5376 86.6 against 74.4,
// 384 x 12288 x 6144 74.3 against 71.8; three ranges of 4 groups, 256 x 18432 x 3072 44.6
// against 39.8; three of 11 and 7, 256 x 18432 x 8192 77.4 against 90.9 and 512 x 8704 x
// 5120 55.7 against 59.5).
constexpr int kNvMinSplitK = 8;
constexpr int kNvMinSplitKFull = 16;
constexpr int kNvMinSplitGroups = 4;
constexpr int kNvHalfSplitTiles = 64;

inline SplitPlan nv_split_plan(int64_t M, int64_t N, int64_t K) {
    SplitPlan sp;
    if (M <= kSkinnyMaxM) return sp;
    const int tiles = static_cast<int>(cdiv(M, kTile) * cdiv(N, kTile));
    const int NG = static_cast<int>(cdiv(K / 2, 128));
    const bool half = tiles <= kNvHalfSplitTiles;
    if (tiles > kTileSlots / 2 || NG < (half ? kNvMinSplitK : kNvMinSplitKFull)) return sp;
    const int units = half ? 2 * tiles : tiles;
    const int S = std::min(kTileSlots / units, NG / kNvMinSplitGroups);
    if (S < (half ? 2 : 3)) return sp;
    sp.ks = static_cast<int>(cdiv(NG, S));
    sp.S = static_cast<int>(cdiv(NG, sp.ks));
    sp.nw = half ? 2 : 4;
    return sp;
}

// one partial tile (or two partial half tiles) per tile and K range
inline int64_t nv_split_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    const SplitPlan sp = nv_split_plan(M, N, K);
    if (sp.S < 2) return 0;
    return cdiv(M, kTile) * cdiv(N, kTile) * sp.S * kPartialBytes;
}

// Small tiles (gemm_mid_nv.h): the first of these whose grid fits the CUs in one round, which
// was the fastest of those that fit on all of 200 measured shapes of 65-1333 rows.  Time (us):
// base + line per 256 elements of K.
struct NvSmallTile {
    int tm, tn;
    double base, line;
};
constexpr NvSmallTile kNvSmall[] = {{64, 64, 5.0, 0.66}, {64, 128, 6.2, 0.8}, {128, 128, 8.5, 1.25}, {128, 192, 11.0, 1.75}};

// Index of the small tile to use, or -1: that estimate against the 256 x 256 kernel's, fitted to
// the same shapes: split-K 14 + 2.6 per group of a K range in half tiles (4.5 in whole tiles),
// half tiles without a split 8.5 + 2.4 per group.  Over 2,780 more shapes of 65-1400 rows the small
// tiles took 0.55 of the time and one of 2,250 choices was more than 3% slower (0.62 per line of 64 x
// 64 tiles chose them for long K too: 200 x 792 x 8704 24.2 against 22.1 us split).  Weight read anew,
// 256 x 13824 x 5120 49.0 -> 39.4 us, 300 x 4096 x 4096 32.7 -> 18.5, 128 x 3072 x 3072 20.7 -> 12.1, 65 x
// 5120 x 2048 21.2 -> 9.8.  Rows that do not start on a cache line (K not a multiple of 256) take 6% longer
// (60 more shapes: 1.08 x the estimate in the mean; 239 x 8824 x 4768 38.6, split-K 37.9).
// At most 64 rows: 64 x 64 or 64 x 128 from 33 rows and N = 8192 on, K up to 8192, and from K = 1024
// on where rows do not start on a cache line (graph-timed against the skinny kernel, weight read anew: 64
// x 24576 x 5120 26.0 / 33.3 us, 33 x 18432 x 3072 16.9 / 20.9, 64 x 12288 x 5120 18.3 / 18.7, 48 x 8192 x
// 3072 12.8 / 12.1; 0.91 in the mean of 1,400 shapes; with 32 rows 32 x 12288 x 3072 12.7 / 11.5, with K =
// 12288 33 x 8192 32.5 / 30.9; 50 x 9232 x 928 8.7 / 7.1 and 1.06 over 190 such shapes).
inline int nv_small_tile(int M, int N, int K, const SplitPlan& sp, int cus) {
    if (M <= kSkinnyMaxM) {
        if (M <= 32 || N < 8192 || K > 8192 || (K % 256 && K < 1024)) return -1;
        return cdiv(N, 64) <= cus ? 0 : cdiv(N, 128) <= cus ? 1 : -1;
    }
    const double groups = static_cast<double>(cdiv(K, 256));
    const double lines = K % 256 ? 1.06 : 1.0;
    for (int i = 0; i < static_cast<int>(sizeof(kNvSmall) / sizeof(kNvSmall[0])); ++i) {
        const NvSmallTile& t = kNvSmall[i];
        if (cdiv(M, t.tm) * cdiv(N, t.tn) > cus) continue;
        const double big = sp.S > 1 ? 14.0 + (sp.nw == 2 ? 2.6 : 4.5) * sp.ks : 8.5 + 2.4 * groups;
        return (t.base + t.line * groups) * lines < big ? i : -1;
    }
    return -1;
}

inline Route nv_route(int M, int N, int K, bool workspace, int cus) {
    Route r;
    r.split = nv_split_plan(M, N, K);
    if (!workspace) r.split.S = 1;
    r.form = nv_small_tile(M, N, K, r.split, cus);
    if (r.form >= 0) {
        r.kind = Route::kSmall;
    } else if (M <= kSkinnyMaxM) {
        r.kind = Route::kSkinny;
        r.form = nv_skinny_form(M, N);
    } else if (r.split.S > 1) {
        r.kind = Route::kSplit;
    } else {
        tile_rounds(r, M, N);
    }
    return r;
}

// ------------------------------------------------------------------ NVFP4 quantizer
// With a given scale, an input padded in rows takes the 16-bit fast path from this many elements
// on.  Below, the general kernel's launch of small workgroups ends sooner than the fast path's of
// up to 1024 threads (graph-timed, general / fast: 230 x 1856 bf16 3.2 / 5.5 us, 1070 x 2048 4.2 /
// 4.6, 1220 x 2688 5.5 / 5.6, 751 x 6976 6.7 / 5.9, 2754 x 7808 22.4 / 11.3; 460 shapes below 4 MB
// 1.4 x in the mean).
constexpr int64_t kNvPadFastElems = 3 << 20;

inline bool nv_quantize_fast_rows(int64_t rows, int64_t orig_rows, int64_t cols) {
    return rows == orig_rows || orig_rows * cols >= kNvPadFastElems;
}

}  // namespace ckh
