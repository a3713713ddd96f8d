// MXFP8 / per-tensor FP8 GEMM on small tiles, one workgroup per CU and one round, for a few
// hundred activation rows (from 17 on in wide layers): grids whose 256 x 256 tiles would leave
// CUs idle.
//
// What bounds it: the rate at which a CU takes in its operand lines.  512 x 5120 x 5120 MXFP8 on 216
// tiles of 128 x 96: 1.18 MB a CU in 24.7 us, 48 GB/s, with the weight in the memory-side cache, and
// in 30.0 us, 39 GB/s, with it read from HBM; 79% of the lines hit the L2 either way, and the matrix
// cores are busy 27% and 20% of the time (counters).  A kernel that only loads reached 57 GB/s per CU
// from HBM with 8 CUs loading, 44-50 with 80 and 23-27 with all 256, where HBM itself is the limit,
// and about 90 from the L2, with loads to registers or to LDS, at any number of loads in flight
// beyond 64 KB.  Lines count, not bytes: with K not a multiple of 128 a row's piece of a stage lies
// in two of them, and a stage takes up to 1.45 x as long.  So a tile's time follows its (TM + TN) K
// operand bytes, about 0.5 us per 128-byte stage of a 128 x 96 tile, and what helps is every CU busy
// with the smallest tile that still fits the grid on the CUs at once; the matrix cores (0.2 us of
// those 0.5) and the prefetch depth (3 to 6 stages measured equal) do not matter.
//
// Against the 256 x 256 kernel's half tiles and split-K (graph-timed MXFP8, us; one weight that stays in
// the caches, then weights read anew): 256 x 9216 x 3072 16.2 / 22.5, 20.5 / 24.1; 512 x 5120 x 5120 23.4
// / 28.8, 29.8 / 30.4; 1024 x 3072 x 3072 16.8 / 25.2, 16.7 / 25.3; 256 x 3072 x 3072 9.1 / 17.5, 9.5 /
// 17.6.  Six layers of 512 x 5120 x 5120 in turn, whose 157 MB the caches partly hold, run level.
//
// A 512-thread workgroup computes a TM x TN tile.  K advances one 128-byte line per row and
// stage; the two K groups of four waves each take one of a stage's two 64-wide MFMA steps, so
// that every SIMD holds two waves whose LDS reads, loads and matrix work overlap, and meet in
// LDS at the end.  Within a group the waves are 4 (m) x 1 (n), or 2 x 2 for 64-row tiles, in
// 32 x 32 MFMA tiles.
//
// Stages move by whole-line direct-to-LDS loads into a ring of NST buffers.  At step t the
// fragments of stage t are in registers, stage t + 1 is resident and read during step t's
// MFMAs, and the loads of stages t + 2 .. t + NST are in flight.  The E8M0 scale words come
// with the stage (256 bytes per wave), so every vector-memory instruction of the loop is a
// direct-to-LDS load and the vmcnt waits count them exactly.  Each of a step's MFMAs sits in a
// slot of its own (sched_barrier) with its share of the next stage's LDS reads and of the
// loads: left to itself, the compiler moved the MFMAs of two steps behind both steps' reads.
//
// LDS rows are 128 bytes; logical 16-byte chunk c of row r sits at c ^ (r & 7) ^ ((r >> 3) & 1)
// (16 consecutive rows of one logical chunk hit 16 distinct bank groups).  Operand layout and
// scale selection are the tile kernel's (gemm_mxfp8.hip).
#pragma once

#include <type_traits>
#include <utility>

#include "ckh_common.h"
#include "skinny.h"

namespace ckh {
namespace mid {

using namespace ckh::sk;

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kRow = 128;       // staged bytes per row and stage
constexpr int kThreads = 512;

struct Args {
    const uint8_t* a;   // activation [M, K]
    const uint8_t* b;   // weight [N, K]
    const uint8_t* sa;  // swizzled E8M0
    const uint8_t* sb;
    const void* bias;   // null: none
    int bias_code;
    void* out;
    int M, N, K;
    int ncb;               // scale column blocks: ceil(K/32/4)
    int sa_rows, sb_rows;  // padded scale rows
    int tiles_m;           // TM x TN tiles along m
    const float* tsa;      // per-tensor mode: the two fp32 tensor scales (device)
    const float* tsb;
};

// Workgroups are dispatched round-robin over the 8 XCDs; XCD x gets the x-th contiguous run of
// the G tiles.
__device__ __forceinline__ int xcd_run(int b, int G) {
    const int x = b & 7;
    return x * (G >> 3) + min(x, G & 7) + (b >> 3);
}

template <int OUT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    return (OUT == CKH_BF16 ? f_to_bf16_rne(a) : f_to_f16(a)) | ((OUT == CKH_BF16 ? f_to_bf16_rne(b) : f_to_f16(b)) << 16);
}

// fn(integral_constant<int, K>) for each K in order
template <typename Fn, int... K>
__device__ __forceinline__ void for_each_index(Fn&& fn, std::integer_sequence<int, K...>) {
    (fn(std::integral_constant<int, K>{}), ...);
}

template <int VM>
__device__ __forceinline__ void wait_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(VM));
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

// finish_tile's sums: K groups 0 and 1 end with them; the first column of a wave's part that
// lane half h of group kg then holds (tiles i and quads q add 32 i + 8 q, and 4 columns follow).
__host__ __device__ constexpr bool holds_sums(int kg) { return kg < 2; }
template <int TN, int WN>
__host__ __device__ constexpr int sum_column(int kg, int wn, int h) {
    return wn * (TN / WN) + 16 * kg + 4 * h;
}

// The end of a tile, in LDS that no load writes any more (at least TM * TN * 2 KG bytes): the sums
// of the KG K groups (of WM x WN waves, wave = WM WN kg + WM wn + wm) added, times alpha
// (SCALE), plus the bias in lds_bias, rounded and stored.  acc: a wave's NT x MT MFMA tiles;
// result lane 32 h + r, register 4 g + e of tile (i, j) holds column 32 i + 8 g + 4 h + e, row
// 32 j + r of the wave's part.
template <int OUT, bool SCALE, int TM, int TN, int KG, int WM, int MT, int NT>
__device__ __forceinline__ void finish_tile(v16f (&acc)[NT][MT], uint8_t* lds, const float* lds_bias, float alpha,
                                            bool bias, void* out, int M, int N, int m0, int n0, int wave, int lane) {
    constexpr int WPG = 8 / KG, WN = WPG / WM, PITCH = TN * 2 + 16;  // staged 16-bit output row
    const int kg = wave / WPG, wig = wave % WPG, wm = wig % WM, wn = wig / WM;
    const int h = lane >> 5, r = lane & 31;
    // The upper half of the groups gives its sums to the lower half, until two are left.
#pragma unroll
    for (int G = KG; G > 2; G /= 2) {
        float4* red = reinterpret_cast<float4*>(lds) + (kg % (G / 2) * WPG + wig) * (MT * NT * 4 * 64) + lane;
        if (kg >= G / 2 && kg < G) {
#pragma unroll
            for (int q = 0; q < MT * NT * 4; ++q) {
                const v16f& a = acc[q / 4 / MT][q / 4 % MT];
                red[q * 64] = make_float4(a[4 * (q % 4)], a[4 * (q % 4) + 1], a[4 * (q % 4) + 2], a[4 * (q % 4) + 3]);
            }
        }
        wait_barrier<63>();
        if (kg < G / 2) {
#pragma unroll
            for (int q = 0; q < MT * NT * 4; ++q) {
                v16f& a = acc[q / 4 / MT][q / 4 % MT];
                const float4 o = red[q * 64];
                a[4 * (q % 4)] += o.x;
                a[4 * (q % 4) + 1] += o.y;
                a[4 * (q % 4) + 2] += o.z;
                a[4 * (q % 4) + 3] += o.w;
            }
        }
        wait_barrier<63>();
    }
    // The last two K groups exchange halves of every MFMA tile (register quads g = 0, 1 and 2, 3):
    // group 0 ends with quads 0, 1, group 1 with 2, 3.
    float4* red = reinterpret_cast<float4*>(lds) + wig * (MT * NT * 4 * 64) + lane;
    auto send = [&](auto g0_c) __attribute__((always_inline)) {
        constexpr int g0 = decltype(g0_c)::value;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int g = g0; g < g0 + 2; ++g)
                    red[((i * MT + j) * 4 + g) * 64] = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1],
                                                                   acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
    };
    if (kg == 0) send(std::integral_constant<int, 2>{});
    else if (kg == 1) send(std::integral_constant<int, 0>{});
    wait_barrier<63>();
    float4 v[NT][MT][2];
    auto recv = [&](auto g0_c) __attribute__((always_inline)) {
        constexpr int g0 = decltype(g0_c)::value;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int g = g0 + q;
                    const float4 o = red[((i * MT + j) * 4 + g) * 64];
                    v[i][j][q] = make_float4(acc[i][j][4 * g] + o.x, acc[i][j][4 * g + 1] + o.y,
                                             acc[i][j][4 * g + 2] + o.z, acc[i][j][4 * g + 3] + o.w);
                }
    };
    if (kg == 0) recv(std::integral_constant<int, 0>{});
    else if (kg == 1) recv(std::integral_constant<int, 2>{});

    const int ml = wm * (TM / WM) + r;             // row of MFMA row tile 0
    const int nl = sum_column<TN, WN>(kg, wn, h);  // column of MFMA column tile 0, quad 0
    // (groups 2 and 3 hold no sums, and their nl would run past the TN columns of lds_bias)
    const bool mine = holds_sums(kg);
    if (mine) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float4 bv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (bias) bv = *reinterpret_cast<const float4*>(lds_bias + nl + 32 * i + 8 * q);
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    float4& o = v[i][j][q];
                    if constexpr (SCALE) o = make_float4(o.x * alpha, o.y * alpha, o.z * alpha, o.w * alpha);
                    if (bias) o = make_float4(o.x + bv.x, o.y + bv.y, o.z + bv.z, o.w + bv.w);
                }
            }
    }
    if constexpr (OUT == CKH_F32) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int m = m0 + ml + 32 * j;
            if (m >= M || !mine) continue;
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int n = n0 + nl + 32 * i + 8 * q;
                    float* o = static_cast<float*>(out) + static_cast<int64_t>(m) * N + n;
                    const float e[4] = {v[i][j][q].x, v[i][j][q].y, v[i][j][q].z, v[i][j][q].w};
                    if (n + 3 < N && (N & 3) == 0) {
                        *reinterpret_cast<float4*>(o) = v[i][j][q];
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (n + k < N) o[k] = e[k];
                    }
                }
        }
    } else {
        // 16-bit output: staged as TM rows in LDS, then whole rows, 16 bytes per lane
        wait_barrier<63>();  // the exchange area is read
        if (mine) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float4 o = v[i][j][q];
                        *reinterpret_cast<uint2*>(lds + (ml + 32 * j) * PITCH + (nl + 32 * i + 8 * q) * 2) =
                            make_uint2(pack2<OUT>(o.x, o.y), pack2<OUT>(o.z, o.w));
                    }
        }
        wait_barrier<63>();
        constexpr int LPR = TN / 8;  // 16-byte pieces per output row
        const bool n8 = (N & 7) == 0;
#pragma unroll
        for (int k = 0; k < TM * LPR / kThreads; ++k) {
            const int piece = k * kThreads + wave * 64 + lane, row = piece / LPR, lr = piece - row * LPR;
            const int n = n0 + 8 * lr;
            const bool vec = n8 && n + 8 <= N;
            const v4u d = *reinterpret_cast<const v4u*>(lds + row * PITCH + lr * 16);
            if (m0 + row >= M) continue;
            uint16_t* o = static_cast<uint16_t*>(out) + static_cast<int64_t>(m0 + row) * N + n;
            if (vec) {
                __builtin_nontemporal_store(d, reinterpret_cast<v4u*>(o));
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (n + e < N) o[e] = static_cast<uint16_t>(d[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}

template <bool UNIT, int TM, int TN, int NST>
struct Shape {
    static constexpr int WM = TM >= 128 ? 4 : 2, WN = 4 / WM;         // waves of a K group along m, n
    static constexpr int MT = TM / WM / 32, NT = TN / WN / 32;        // 32 x 32 MFMA tiles per wave
    static_assert(MT * WM * 32 == TM && NT * WN * 32 == TN, "whole MFMA tiles");
    static constexpr int AL = TM / 64, BL = (TN + 63) / 64;           // code loads per wave and stage
    static constexpr int LPW = AL + BL + (UNIT ? 0 : 1);              // loads per wave and stage
    static constexpr int CODES = (AL + BL) * 8192;         // (TN = 96: the last 32 rows stay zero)
    static constexpr int STG = CODES + (UNIT ? 0 : 2048);  // + scale words: 1 KB per operand
    static_assert(TM * TN * 4 <= NST * STG && TM * (TN * 2 + 16) <= NST * STG, "the epilogue reuses the ring");
    static_assert((NST - 1) * LPW < 64, "vmcnt range");
};

template <int OUT, bool UNIT, int TM, int TN, int NST>
__global__ __launch_bounds__(kThreads) void gemm_mid_kernel(Args p) {
    using S = Shape<UNIT, TM, TN, NST>;
    constexpr int MT = S::MT, NT = S::NT, LPW = S::LPW, STG = S::STG, AL = S::AL, BL = S::BL;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NST * STG];
    __shared__ __attribute__((aligned(16))) float lds_bias[TN];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave >> 2, wm = wave & (S::WM - 1), wn = (wave & 3) / S::WM;
    const int h = lane >> 5, r = lane & 31;

    // m fastest: tiles that share a weight panel run side by side on one XCD
    const int idx = xcd_run(blockIdx.x, gridDim.x);
    const int m0 = idx % p.tiles_m * TM, n0 = idx / p.tiles_m * TN;
    const int t1 = (p.K + kRow - 1) / kRow;  // stages

    uint32_t bias_bits = 0;
    if (p.bias && tid < TN) bias_bits = load_bias_bits(p.bias, p.bias_code, n0 + tid, p.N);

    const __amdgpu_buffer_rsrc_t ra =
        buffer_rsrc(p.a + static_cast<int64_t>(m0) * p.K, static_cast<uint32_t>(min(TM, p.M - m0)) * p.K);
    const __amdgpu_buffer_rsrc_t rb =
        buffer_rsrc(p.b + static_cast<int64_t>(n0) * p.K, static_cast<uint32_t>(min(TN, p.N - n0)) * p.K);
    const __amdgpu_buffer_rsrc_t rsa = buffer_rsrc(p.sa, UNIT ? 0u : static_cast<uint32_t>(p.sa_rows) * p.ncb * 4);
    const __amdgpu_buffer_rsrc_t rsb = buffer_rsrc(p.sb, UNIT ? 0u : static_cast<uint32_t>(p.sb_rows) * p.ncb * 4);

    // Load q = wave + 8 i of a stage fills rows 8 q .. 8 q + 7 of the stage (activation rows, then
    // weight rows), lane l physical chunk l % 8 of row 8 q + l / 8.
    const int cb = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) << 4;
    const uint32_t voff = static_cast<uint32_t>((wave * 8 + (lane >> 3)) * p.K + cb);
    const uint32_t rowstep = 64u * p.K;
    // scale words: 512-byte chunk (128-row block, stage) of the swizzled tensor, two blocks
    // per operand (a 96-, 160- or 192-wide tile's weight rows can straddle two); wave w loads quarter w % 4 of the
    // activation's (w < 4) or the weight's 1 KB
    const int sq = (wave & 3) * 64 + lane;  // word of the operand's two blocks
    const __amdgpu_buffer_rsrc_t rs = wave < 4 ? rsa : rsb;
    const uint32_t soff = static_cast<uint32_t>((((wave < 4 ? m0 : n0) >> 7) + (sq >> 7)) * p.ncb * 512 + (sq & 127) * 4);
    auto issue_part = [&](int t, uint8_t* dst, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < AL + BL) {
            constexpr bool act = i < AL;
            const uint32_t o = t * kRow + cb < p.K ? voff + static_cast<uint32_t>(t * kRow) : 0x80000000u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(act ? ra : rb, (lds_void*)(dst + (wave + 8 * i) * 1024), 16,
                                                     o + (act ? i : i - AL) * rowstep, 0, 0, 0);
        } else {
            const uint32_t so = t < p.ncb ? soff + static_cast<uint32_t>(t * 512) : 0x80000000u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(dst + S::CODES + wave * 256), 4, so, 0, 0, 0);
        }
    };

    // One stage's operands of this wave: rows 32 t + r of its part, bytes 64 kg + 16 h .. and
    // 64 kg + 32 + 16 h .. of the line, and the rows' scale words.
    struct Frags {
        v8i a[MT], b[NT];
        uint32_t sa[MT], sb[NT];
    };
    const int x = swz8(r);
    const uint32_t lo = static_cast<uint32_t>(((4 * kg + h) ^ x) << 4), hi = static_cast<uint32_t>(((4 * kg + 2 + h) ^ x) << 4);
    const uint32_t arow = static_cast<uint32_t>((wm * (TM / S::WM) + r) * kRow);
    const uint32_t brow = static_cast<uint32_t>((TM + wn * (TN / S::WN) + r) * kRow);
    // scale word of row 32 t + r of the wave's part: the staged block of its 128 rows, chunk r,
    // word (row % 128) / 32
    const int am = (m0 & 127) + wm * (TM / S::WM), bn = (n0 & 127) + wn * (TN / S::WN);
    auto word_at = [](int row) { return static_cast<uint32_t>((row >> 7) * 512 + ((row & 127) >> 5) * 4); };
    const int sh = 8 * (2 * kg + h);
    auto frag = [&](const uint8_t* row) __attribute__((always_inline)) {
        const v4u u = *reinterpret_cast<const v4u*>(row + lo), w = *reinterpret_cast<const v4u*>(row + hi);
        return v8i{(int)u[0], (int)u[1], (int)u[2], (int)u[3], (int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    };
    // Read I of a stage: scale words, then weight and activation fragments
    constexpr int NREAD = 1 + NT + MT;
    auto read_part = [&](const uint8_t* s, Frags& F, auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value;
        if constexpr (I == 0) {
            if constexpr (!UNIT) {
                const uint8_t* w = s + S::CODES + r * 16;
#pragma unroll
                for (int t = 0; t < MT; ++t) F.sa[t] = *reinterpret_cast<const uint32_t*>(w + word_at(am + 32 * t));
#pragma unroll
                for (int t = 0; t < NT; ++t) F.sb[t] = *reinterpret_cast<const uint32_t*>(w + 1024 + word_at(bn + 32 * t));
            }
        } else if constexpr (I <= NT) {
            F.b[I - 1] = frag(s + brow + (I - 1) * 32 * kRow);
        } else {
            F.a[I - 1 - NT] = frag(s + arow + (I - 1 - NT) * 32 * kRow);
        }
    };

    v16f acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = v16f{};
    auto mfma = [&](const Frags& F, auto k_c) __attribute__((always_inline)) {
        constexpr int i = decltype(k_c)::value / MT, j = decltype(k_c)::value % MT;
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            F.b[i], F.a[j], acc[i][j], 0, 0, 0, UNIT ? 0x7f7f7f7fu : F.sb[i] >> sh, 0, UNIT ? 0x7f7f7f7fu : F.sa[j] >> sh);
    };

    // (A loop, not unrolled: where the compiler sees loads write a known part of `lds`, it drains
    // every load in flight before the next LDS read.)
    uint8_t* cur = lds;  // buffer of stage t
#pragma unroll 1
    for (int s = 0; s < NST; ++s, cur += STG)
        for_each_index([&](auto i_c) { issue_part(s, cur, i_c); }, std::make_integer_sequence<int, LPW>{});
    wait_barrier<(NST - 1) * LPW>();
    cur -= NST * STG;
    Frags F0, F1;
    for_each_index([&](auto i_c) { read_part(cur, F0, i_c); }, std::make_integer_sequence<int, NREAD>{});
    // One step: the MFMAs of stage t (fragments F), each in a slot with its share of stage
    // t + 1's reads (into G) and of the loads of stage t + NST (into stage t's buffer)
    constexpr int SLOTS = MT * NT, ACTS = NREAD + LPW;
    auto step = [&](int t, const Frags& F, Frags& G) __attribute__((always_inline)) {
        wait_barrier<(NST - 2) * LPW>();  // stage t + 1 resident, stage t read by all
        uint8_t* nx = cur + STG == lds + NST * STG ? lds : cur + STG;
        for_each_index([&](auto k_c) {
            constexpr int k = decltype(k_c)::value, a0 = k * ACTS / SLOTS, a1 = (k + 1) * ACTS / SLOTS;
            mfma(F, k_c);
            for_each_index([&](auto d_c) {
                constexpr int act = a0 + decltype(d_c)::value;
                if constexpr (act < NREAD) read_part(nx, G, std::integral_constant<int, act>{});
                else issue_part(t + NST, cur, std::integral_constant<int, act - NREAD>{});
            }, std::make_integer_sequence<int, a1 - a0>{});
            __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, SLOTS>{});
        cur = nx;
    };
    int t = 0;
    for (; t + 1 < t1; t += 2) {
        step(t, F0, F1);
        step(t + 1, F1, F0);
    }
    if (t < t1) for_each_index([&](auto k_c) { mfma(F0, k_c); }, std::make_integer_sequence<int, SLOTS>{});
    if (p.bias && tid < TN) lds_bias[tid] = bias_value(bias_bits, p.bias_code);
    wait_barrier<0>();  // trailing loads have landed and every read is done: LDS is free

    finish_tile<OUT, UNIT, TM, TN, 2, S::WM, MT, NT>(acc, lds, lds_bias, UNIT ? p.tsa[0] * p.tsb[0] : 1.0f,
                                                  p.bias != nullptr, p.out, p.M, p.N, m0, n0, wave, lane);
}

}  // namespace mid
}  // namespace ckh
