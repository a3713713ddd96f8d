// NVFP4 GEMM on small tiles, one workgroup per CU and one round: the counterpart of gemm_mid.h
// for grids whose 256 x 256 tiles would leave CUs idle.
//
// A 512-thread workgroup computes a TM x TN tile; K advances one 128-byte line per row and
// step (256 elements, four 64-element stages dealt to KG K groups of waves).  Packed codes and
// scale words come to LDS by direct-to-LDS loads into a ring of NST lines, and are decoded to
// fp16 in registers one 16-wide MFMA substep ahead of the MFMAs, each MFMA in a slot
// (sched_barrier) with its share of the decode, of the next stage's LDS reads and of the loads,
// as in the 256 x 256 kernel (gemm_nvfp4.hip: arithmetic, operand layout and chunk swizzle are
// its).  Two waves share each SIMD, so one's decode fills the other's waits.
//
// What bounds it: the decode, four converts and four packed multiplies per 32-row operand tile
// and 16-wide substep.  More K groups of fewer waves give each wave a larger part of the tile
// and so fewer decodes per MFMA: 128 x 128 with 2 groups (64 x 64 a wave) spends 8 decode
// instructions per MFMA and took 46.1 us on 256 x 13824 x 5120, with 4 groups (128 x 64 a wave)
// 6 and 41.9 us; with all codes zero, i.e. without the power limit, 35.4.  (On another card, with the
// weight kept in the caches / read anew: 37.0 / 39.4, the 256 x 256 kernel's split-K 45.2 / 49.0; the
// matrix cores are busy 46% of the time.)
#pragma once

#include "gemm_mid.h"
#include "quant_math.h"

namespace ckh {
namespace midnv {

using namespace ckh::mid;

struct Args {
    const uint8_t* a;   // packed E2M1 [M, K / 2]
    const uint8_t* b;   // [N, K / 2]
    const uint8_t* sa;  // swizzled E4M3
    const uint8_t* sb;
    const float* alpha;    // tensor scale, or the activation's
    const float* alpha_b;  // the weight's (null: alpha is the product)
    const void* bias;  // null: none
    int bias_code;
    void* out;
    int M, N, K;           // K in elements
    int ncb;               // scale word columns: ceil(K/16/4)
    int sa_rows, sb_rows;  // padded scale rows
    int tiles_m;           // TM x TN tiles along m
};

// KG K groups of 8 / KG waves: the waves of a group split the tile 2 (m) x 2 (n) with 2 groups
// and 1 x 2 with 4.  A line's four 64-element stages are dealt to the groups in order.
template <int TM, int TN, int KG, int NST>
struct Shape {
    static_assert(KG == 2 || KG == 4, "K groups");
    static constexpr int WM = KG == 2 ? 2 : 1, WN = 2;        // waves of a group
    static constexpr int MT = TM / WM / 32, NT = TN / WN / 32;        // 32 x 32 MFMA tiles per wave
    static constexpr int UPL = 4 / KG;                        // stages of a group per line
    static constexpr int AL = TM / 64, BL = TN / 64;          // code loads per wave and line
    static constexpr int SA = 1, SB = TN > 128 ? 2 : 1;       // staged 128-row scale blocks
    static constexpr int LPW = AL + BL + SA + SB;             // loads per wave and line
    static constexpr int CODES = (TM + TN) * kRow;
    static constexpr int STG = CODES + (SA + SB) * 2048;
    static_assert(TM <= 128 && TM * TN * 2 * KG <= NST * STG && TM * (TN * 2 + 16) <= NST * STG, "the epilogue reuses the ring");
    static_assert((NST - 1) * LPW < 64, "vmcnt range");
};

template <int OUT, int TM, int TN, int KG, int NST>
__global__ __launch_bounds__(kThreads) void gemm_mid_nv_kernel(Args p) {
    using S = Shape<TM, TN, KG, NST>;
    constexpr int WPG = 8 / KG, MT = S::MT, NT = S::NT, AL = S::AL, BL = S::BL, LPW = S::LPW, STG = S::STG;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NST * STG];
    __shared__ __attribute__((aligned(16))) float lds_bias[TN];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / WPG, wig = wave % WPG, wm = wig % S::WM, wn = wig / S::WM;
    const int h = lane >> 5, r = lane & 31;
    const int Kb = p.K / 2;  // code bytes per row

    // m fastest: tiles that share a weight panel run side by side on one XCD
    const int idx = xcd_run(blockIdx.x, gridDim.x);
    const int m0 = idx % p.tiles_m * TM, n0 = idx / p.tiles_m * TN;
    const int t1 = (Kb + kRow - 1) / kRow;  // lines

    uint32_t bias_bits = 0;
    if (p.bias && tid < TN) bias_bits = load_bias_bits(p.bias, p.bias_code, n0 + tid, p.N);

    const __amdgpu_buffer_rsrc_t ra =
        buffer_rsrc(p.a + static_cast<int64_t>(m0) * Kb, static_cast<uint32_t>(min(TM, p.M - m0)) * Kb);
    const __amdgpu_buffer_rsrc_t rb =
        buffer_rsrc(p.b + static_cast<int64_t>(n0) * Kb, static_cast<uint32_t>(min(TN, p.N - n0)) * Kb);
    const __amdgpu_buffer_rsrc_t rsa = buffer_rsrc(p.sa, static_cast<uint32_t>(p.sa_rows) * p.ncb * 4);
    const __amdgpu_buffer_rsrc_t rsb = buffer_rsrc(p.sb, static_cast<uint32_t>(p.sb_rows) * p.ncb * 4);

    // Code load q = wave + 8 i fills rows 8 q .. 8 q + 7 of the line buffer (activation rows, then
    // weight rows), lane l physical chunk l % 8 of row 8 q + l / 8.
    const int cb = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) << 4;
    const uint32_t voff = static_cast<uint32_t>((wave * 8 + (lane >> 3)) * Kb + cb);
    const uint32_t rowstep = 64u * Kb;
    // Scale load: 256-byte half wave % 2 of column wave / 2 (of the line's four) of one 128-row
    // block's 512-byte chunks
    const int scol = wave >> 1;
    const uint32_t soff = static_cast<uint32_t>(scol * 512 + (wave & 1) * 256 + lane * 4);
    auto issue_part = [&](int t, uint8_t* dst, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < AL + BL) {
            constexpr bool act = i < AL;
            const uint32_t o = t * kRow + cb < Kb ? voff + static_cast<uint32_t>(t * kRow) : 0x80000000u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(act ? ra : rb, (lds_void*)(dst + (wave + 8 * i) * 1024), 16,
                                                     o + (act ? i : i - AL) * rowstep, 0, 0, 0);
        } else {
            constexpr int u = i - AL - BL;  // block: the activation's, then the weight's
            const int blk = u < S::SA ? (m0 >> 7) + u : (n0 >> 7) + u - S::SA;
            const uint32_t so =
                4 * t + scol < p.ncb ? static_cast<uint32_t>((blk * p.ncb + 4 * t) * 512) + soff : 0x80000000u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(u < S::SA ? rsa : rsb,
                                                     (lds_void*)(dst + S::CODES + u * 2048 + wave * 256), 4, so, 0, 0, 0);
        }
    };

    // One stage's raw operands: per tile row 32 t + r the lane's 16 code bytes (dword KK for
    // substep KK) and the row's scale word; and one substep's decoded operands.
    struct Raw {
        v4u a[MT], b[NT];
        uint32_t wa[MT], wb[NT];
    };
    struct Dec {
        v8h a[MT], b[NT];
    };
    const int x = swz8(r);
    const uint32_t arow = static_cast<uint32_t>((wm * (TM / S::WM) + r) * kRow);
    const uint32_t brow = static_cast<uint32_t>((TM + wn * (TN / S::WN) + r) * kRow);
    const int am = (m0 & 127) + wm * (TM / S::WM), bn = (n0 & 127) + wn * (TN / S::WN);
    auto word_at = [](int row) { return static_cast<uint32_t>((row >> 7) * 2048 + ((row & 127) >> 5) * 4); };
    constexpr int NREAD = MT + NT;
    // Read I (tile I of the activation, then of the weight) of stage kg UPL + u of a line
    auto read_part = [&](const uint8_t* line, auto u_c, Raw& R, auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value;
        const int st = kg * S::UPL + decltype(u_c)::value;
        const uint32_t chunk = static_cast<uint32_t>(((2 * st + h) ^ x) << 4);
        const uint8_t* w = line + S::CODES + st * 512 + r * 16;
        if constexpr (I < MT) {
            R.a[I] = *reinterpret_cast<const v4u*>(line + arow + I * 32 * kRow + chunk);
            R.wa[I] = *reinterpret_cast<const uint32_t*>(w + word_at(am + 32 * I));
        } else {
            R.b[I - MT] = *reinterpret_cast<const v4u*>(line + brow + (I - MT) * 32 * kRow + chunk);
            R.wb[I - MT] = *reinterpret_cast<const uint32_t*>(w + S::SA * 2048 + word_at(bn + 32 * (I - MT)));
        }
    };
    const int sh = 16 * h;  // the lane's two block scales in its word
    // Part P of decoding substep KK of R into D: half P & 1 (two converts, two multiplies) of
    // activation tile P / 2, then of the weight's
    constexpr int NDEC = 2 * (MT + NT);
    auto decode_part = [&](const Raw& R, auto kk_c, Dec& D, auto p_c) __attribute__((always_inline)) {
        constexpr int KK = decltype(kk_c)::value, P = decltype(p_c)::value, t = P >> 1, hf = P & 1;
        constexpr bool A = t < MT;
        const v2h pr = scale_pair(A ? R.wa[A ? t : 0] : R.wb[A ? 0 : t - MT], sh);
        const v2h sc = KK < 2 ? v2h{pr[0], pr[0]} : v2h{pr[1], pr[1]};
        const uint32_t w = A ? R.a[A ? t : 0][KK] : R.b[A ? 0 : t - MT][KK];
        const v2h e0 = decode2<2 * hf>(w, sc), e1 = decode2<2 * hf + 1>(w, sc);
        v8h& d = A ? D.a[A ? t : 0] : D.b[A ? 0 : t - MT];
        d[4 * hf] = e0[0];
        d[4 * hf + 1] = e0[1];
        d[4 * hf + 2] = e1[0];
        d[4 * hf + 3] = e1[1];
    };

    v16f acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = v16f{};

    // One substep: MT NT MFMAs on Dc, each in a slot with its share of the decode of (Rd, KKd)
    // into Dn and of this substep's extra actions
    constexpr int SLOTS = MT * NT;
    auto substep = [&](const Dec& Dc, const Raw& Rd, auto kkd_c, Dec& Dn, auto nact_c, auto act) __attribute__((always_inline)) {
        constexpr int NACT = decltype(nact_c)::value;
        for_each_index([&](auto k_c) {
            constexpr int k = decltype(k_c)::value, i = k / MT, j = k % MT;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Dc.b[i], Dc.a[j], acc[i][j], 0, 0, 0);
            constexpr int d0 = k * NDEC / SLOTS, d1 = (k + 1) * NDEC / SLOTS;
            for_each_index([&](auto d_c) { decode_part(Rd, kkd_c, Dn, std::integral_constant<int, d0 + decltype(d_c)::value>{}); },
                           std::make_integer_sequence<int, d1 - d0>{});
            constexpr int a0 = k * NACT / SLOTS, a1 = (k + 1) * NACT / SLOTS;
            for_each_index([&](auto a_c) { act(std::integral_constant<int, a0 + decltype(a_c)::value>{}); },
                           std::make_integer_sequence<int, a1 - a0>{});
            __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, SLOTS>{});
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    auto none = [](auto) {};

    // (a loop, not unrolled: see gemm_mid.h)
    uint8_t* cur = lds;  // buffer of line t
#pragma unroll 1
    for (int s = 0; s < NST; ++s, cur += STG)
        for_each_index([&](auto i_c) { issue_part(s, cur, i_c); }, std::make_integer_sequence<int, LPW>{});
    wait_barrier<(NST - 1) * LPW>();
    cur -= NST * STG;
    Raw R0, R1;
    Dec D0, D1;
    for_each_index([&](auto i_c) { read_part(cur, C0{}, R0, i_c); }, std::make_integer_sequence<int, NREAD>{});
    for_each_index([&](auto p_c) { decode_part(R0, C0{}, D0, p_c); }, std::make_integer_sequence<int, NDEC>{});

    // One stage: its four substeps on R (decoded one ahead), the group's next stage (stage u of its
    // line) read into Rn during the first and its first substep decoded during the last.  The
    // stage that reads the next line (NEXT) first waits for it and, line t then being read by
    // all, loads line t + NST into line t's buffer.
    auto stage = [&](int t, auto u_c, auto next_c, const Raw& R, Raw& Rn) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(next_c)::value;
        uint8_t* nx = cur;
        if constexpr (NEXT) {
            wait_barrier<(NST - 2) * LPW>();
            nx = cur + STG == lds + NST * STG ? lds : cur + STG;
        }
        auto reads = [&](auto i_c) __attribute__((always_inline)) { read_part(nx, u_c, Rn, i_c); };
        auto loads = [&](auto i_c) __attribute__((always_inline)) { issue_part(t + NST, cur, i_c); };
        using CL = std::integral_constant<int, NEXT ? LPW : 0>;
        substep(D0, R, C1{}, D1, std::integral_constant<int, NREAD>{}, reads);
        substep(D1, R, C2{}, D0, CL{}, loads);
        substep(D0, R, C3{}, D1, C0{}, none);
        substep(D1, Rn, C0{}, D0, C0{}, none);
        cur = nx;
    };
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;
    if constexpr (S::UPL == 2) {
        for (int t = 0; t < t1; ++t) {
            stage(t, C1{}, No{}, R0, R1);   // the group's stage 0 of line t, reading stage 1
            stage(t, C0{}, Yes{}, R1, R0);  // stage 1, reading stage 0 of line t + 1
        }
    } else {
        int t = 0;
        for (; t + 1 < t1; t += 2) {
            stage(t, C0{}, Yes{}, R0, R1);
            stage(t + 1, C0{}, Yes{}, R1, R0);
        }
        if (t < t1) stage(t, C0{}, Yes{}, R0, R1);
    }
    if (p.bias && tid < TN) lds_bias[tid] = bias_value(bias_bits, p.bias_code);
    wait_barrier<0>();  // trailing loads have landed and every read is done: LDS is free
    finish_tile<OUT, true, TM, TN, KG, S::WM, MT, NT>(acc, lds, lds_bias, tensor_scale(p.alpha, p.alpha_b), p.bias != nullptr, p.out, p.M, p.N, m0,
                                              n0, wave, lane);
}

}  // namespace midnv
}  // namespace ckh
