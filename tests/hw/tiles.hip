// Host-side facts about the small-tile GEMMs, from the kernels' own headers.  TEST CODE ONLY:
// built into tests/hw/libckh_hwcheck.so; nothing here runs on a GPU.
#include <algorithm>

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
