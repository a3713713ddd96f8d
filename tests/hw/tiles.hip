// Host-side facts about the GEMMs, from the kernels' own headers: the kernel that a call's sizes
// select, and the small tiles' bias columns.  TEST CODE ONLY: built into
// tests/hw/libckh_hwcheck.so; nothing here runs on a GPU.
#include <algorithm>

#include "dispatch.h"
#include "gemm_mid.h"
#include "gemm_mid_nv.h"

using namespace ckh;

namespace {

// One past the last bias column that any wave of a tile reads (finish_tile).
template <int TN, int KG, int WN, int NT>
int bias_end() {
    int end = 0;
    for (int kg = 0; kg < KG; ++kg)
        for (int wn = 0; wn < WN; ++wn)
            for (int h = 0; h < 2; ++h)
                if (mid::holds_sums(kg)) end = std::max(end, mid::sum_column<TN, WN>(kg, wn, h) + 32 * (NT - 1) + 8 + 4);
    return end;
}

template <int TM, int TN, int NST>
int mx_bias_end() {
    using S = mid::Shape<false, TM, TN, NST>;
    return bias_end<TN, 2, S::WN, S::NT>();
}

template <int TM, int TN, int KG, int NST>
int nv_bias_end() {
    using S = midnv::Shape<TM, TN, KG, NST>;
    return bias_end<TN, KG, S::WN, S::NT>();
}

}  // namespace

// bias_end of the MXFP8 / FP8 (nv 0) or NVFP4 (nv 1) small tile tm x tn; 0: no such tile.
extern "C" int ckh_tile_bias_end(int nv, int tm, int tn) {
#define MX(M, N, S) if (!nv && tm == M && tn == N) return mx_bias_end<M, N, S>()
#define NV(M, N, G, S) if (nv && tm == M && tn == N) return nv_bias_end<M, N, G, S>()
    MX(64, 64, 6);
    MX(128, 64, 5);
    MX(128, 96, 4);
    MX(128, 128, 4);
    MX(128, 160, 3);
    MX(128, 192, 3);
    MX(64, 128, 5);
    NV(64, 64, 4, 6);
    NV(64, 128, 4, 5);
    NV(128, 128, 4, 4);
    NV(128, 192, 2, 3);
#undef MX
#undef NV
    return 0;
}

// The kernel that serves a GEMM call on a device of `cus` CUs: fills out[0..5] and returns
//   0 skinny     waves, weight tiles, activation tiles, staged or decoded activation rows, code rows
//   1 small tile rows, columns
//   2 split-K    ranges, stages (MXFP8, FP8) or groups (NVFP4) per range, 4 whole / 2 half tiles
//   3 tiles      whole tiles, tiles run as two halves, weight-prefetch workgroups
extern "C" int ckh_route(int nv, int64_t M, int64_t N, int64_t K, int workspace, int cus, int* out) {
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
    const Route r = nv ? nv_route(m, n, k, workspace != 0, cus) : mx_route(m, n, k, workspace != 0, cus);
    std::fill(out, out + 6, 0);
    if (r.kind == Route::kSkinny) {
        const SkinnyForm f = nv ? kNvSkinny[r.form] : kMxSkinny[r.form];
        out[0] = f.waves, out[1] = f.weight_tiles, out[2] = f.act_tiles, out[3] = f.act_rows, out[4] = f.code_rows;
    } else if (r.kind == Route::kSmall) {
        out[0] = nv ? kNvSmall[r.form].tm : kMxSmall[r.form].tm;
        out[1] = nv ? kNvSmall[r.form].tn : kMxSmall[r.form].tn;
    } else if (r.kind == Route::kSplit) {
        out[0] = r.split.S, out[1] = r.split.ks, out[2] = r.split.nw;
    } else {
        out[0] = r.n_full, out[1] = r.n_half, out[2] = r.n_pref;
    }
    return r.kind;
}

// Number of skinny forms of a format.
extern "C" int ckh_skinny_forms(int nv) {
    return nv ? static_cast<int>(sizeof(kNvSkinny) / sizeof(kNvSkinny[0]))
              : static_cast<int>(sizeof(kMxSkinny) / sizeof(kMxSkinny[0]));
}

// Whether the NVFP4 quantizer with a given scale may take its fast path for this row padding.
extern "C" int ckh_nv_quantize_fast_rows(int64_t rows, int64_t orig_rows, int64_t cols) {
    return nv_quantize_fast_rows(rows, orig_rows, cols);
}
