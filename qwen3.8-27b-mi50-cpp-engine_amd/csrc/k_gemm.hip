// k_gemm.hip -- prefill ingest on int8 MFMA: the per-(row, group) W8A8 GEMM of the reference's
// layer-split prefill and its two quantizers, as hand-written gfx950 kernels.
//
// Reference: one rocBLAS int8 gemm_ex per K group writes an int32 slab (src/q27_rb.cpp:43-55), and
// an epilogue sums the slabs with the product of the two scales (src/q27_epi.hip:189-203, fp32 +
// residual form 235-243). The groups are GS = 1024 columns (or the whole K); weights are the
// per-64 mirror requantized per (row, group) (src/q27_epi.hip:14-35), activations are quantized
// per (token, group) (q27_quant_group, src/q27_epi.hip:64-75).
//
// Semantics kept bit for bit:
//   weights:     sg = max of the group's per-64 scales; inv = sg > 0 ? 1/sg : 0;
//                code = clamp(rint(((float)w * s64) * inv), -127, 127)
//   activations: sc = max|v| * (1/127); qi = sc > 0 ? 1/sc : 0; code = clamp(rint(v * qi), -127, 127)
//   GEMM:        acc_g = exact int32 dot over group g; o = 0;
//                for g ascending: o = fmaf((float)acc_g, sw[n][g] * sx[t][g], o);
//                y[t][n] = o * alpha (+ rs * res[t][n])
// The int32 group sums do not depend on the order of their terms, so the MFMA tiling cannot
// change them; the fp32 part runs per output in the reference's group order.
//
// GEMM tiling: a launch takes the cheapest of a list of forms (pick_form): k_gemm_i8g_ring (64 to 256 tokens
// x 64 to 256 weight rows per block, 128-byte K stages in an LDS ring), k_gemm_i8g_sk (few tokens: small tiles whose
// waves split K), k_gemm_i8g_w4 (256 x 256 tiles, one group over K) and k_gemm_i8g_rs (256 x 128, several groups). At
// the end of each group the int32 tiles are folded into fp32 accumulators with the group's scales and restarted
// from zero. The general form, k_gemm_i8g, takes the other shapes and some with several small groups: a 256-thread
// block computes a 128-token x 128-row tile; wave w owns the 64 x 64 quarter (w / 2, w % 2) as 2 x 2 v_mfma_i32_32x32x32_i8 tiles, and two blocks share a
// CU. K advances 64 bytes per stage through a ring of 4 LDS stages (3 when the scales of 17+ groups take the room)
// filled by LDS DMA ahead of the multiply.
#include <math.h>
#include <stdlib.h>
#include <mutex>
#include <type_traits>

#include "q27x_dev.h"
#include "q27x_int.h"

namespace q27x {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kGN = 128, kGK = 64;                // block tile: BM tokens x 128 weight rows, 64 K bytes per stage
constexpr int kSkLds = 160 * 1024;                 // LDS of the split-K kernel
constexpr int kGMaxG = 20;                         // groups per row held in LDS (K / GS)
template <int BM, int NS> struct GemmCfg {
    static constexpr int S = NS;                   // stages in the LDS ring
    static constexpr int NW = BM / 32;             // waves: BM / 64 token rows x 2 weight columns of 64
    static constexpr int Stage = (BM + kGN) * kGK; // bytes per stage: A rows, then B rows
    static constexpr int NI = Stage / (1024 * NW); // 1 KiB transfers per wave per stage
    static_assert(Stage % (1024 * NW) == 0, "whole transfers per wave");
};

struct GemmArgs {
    const int8_t* w;    // [N][K] per-(row, group) codes
    const float* sw;    // [N][ng]
    const int8_t* x;    // [M][K] per-(token, group) codes
    const float* sx;    // [M][ng]
    float* y;           // [M][ldy] (bf16 when out_bf16)
    const float* res;   // [M][ldr] or null (bf16 when res_bf16)
    float alpha, rs;
    int M, N, K, gs, ng, ldy, ldr;
    int out_bf16, res_bf16;
    AlphaSel asel;
};

template <int BM, int NS>
__global__ __launch_bounds__(BM * 2) void k_gemm_i8g(GemmArgs a) {
    constexpr int kGS = GemmCfg<BM, NS>::S, kGStage = GemmCfg<BM, NS>::Stage, NI = GemmCfg<BM, NS>::NI;
    constexpr int kGM = BM, BN = kGN, NT = BM * 2;
    constexpr int JT = 2;                          // 32-row weight tiles per wave
    __shared__ __align__(16) int8_t sR[kGS * kGStage];
    // the block's scales, [row][ng] floats: 128 token rows, then BN weight rows (dynamic LDS,
    // sized by the launch to the group count, so short K leaves room for a deeper ring)
    extern __shared__ float sScl[];
    float* sSx = sScl;
    float* sSw = sScl + kGM * a.ng;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;       // wave tile: tokens 64 wm .., weight rows (BN / 2) wn ..
    // Tile order. Blocks are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8), and each
    // XCD has its own L2; block b therefore takes tile (b % 8) * T/8 + b / 8 of a grouped order
    // (groups of 4 token tiles, weight tile major within a group), so each XCD streams one
    // contiguous run of that order: with 32 token tiles, its own 4 token tiles (kept in its L2)
    // against every weight tile, and the 32 blocks it runs at once share 4 token tiles and 8
    // weight tiles. When T is not a multiple of 8 the order is the plain one.
    const int nt = a.N / BN, mt = (a.M + kGM - 1) / kGM, T = nt * mt;
    const int b = blockIdx.x;
    const int tile = (T % 8 == 0) ? (b % 8) * (T / 8) + b / 8 : b;
    const int grp = tile / (4 * nt), fm = grp * 4, gsz = (mt - fm < 4) ? mt - fm : 4;
    const int within = tile - grp * 4 * nt;
    const int m0 = (fm + within % gsz) * kGM, n0 = (within / gsz) * BN;
    const int K = a.K, ng = a.ng, spg = a.gs / kGK, nsteps = K / kGK;

    // Stage layout: rows of 64 bytes, A rows 0..BM-1 then B rows 0..BN-1; chunk c (16 bytes) of row
    // R sits in slot c ^ ((R >> 2) & 3) of its row, so the 16 consecutive rows one operand read
    // serves at a time (same c) fill the 16 distinct 16-byte positions of a 256-byte bank window
    // (SQ_LDS_BANK_CONFLICT reads 0; with (R >> 1) & 3 it was 17% of busy cycles). DMA: instruction i (< NI) of wave
    // w fills stage bytes 1 KiB (NI w + i) .. +1 KiB = stage rows 16 (NI w + i) .. +16; lane l writes
    // row 16 (NI w + i) + l / 4, slot l % 4, so it loads that row's chunk (l % 4) ^ ((row >> 2) & 3).
    const int8_t* gp[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int rs = 16 * (NI * wave + i) + (lane >> 2);         // stage row
        const int r = rs < kGM ? rs : rs - kGM;
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        if (rs < kGM) {
            const int t = (m0 + r < a.M) ? m0 + r : a.M - 1;       // rows past M repeat row M - 1
            gp[i] = a.x + (size_t)t * K + 16 * c;
        } else {
            gp[i] = a.w + (size_t)(n0 + r) * K + 16 * c;
        }
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sR;
    auto issue = [&](int step, int slot) __attribute__((always_inline)) {
        const uint32_t base = lds0 + slot * kGStage + 1024 * NI * wave;
#pragma unroll
        for (int i = 0; i < NI; ++i) lds_dma16(gp[i] + step * kGK, __builtin_amdgcn_readfirstlane(base + 1024 * i));
    };

    // the first stages, then the block's scales for every group (rows past M read row M - 1;
    // their outputs are not stored)
#pragma unroll
    for (int p = 0; p < kGS - 1; ++p) issue(p < nsteps ? p : 0, p);
    for (int i = tid; i < kGM * ng; i += NT) {
        const int r = i / ng, g = i - r * ng;
        const int t = (m0 + r < a.M) ? m0 + r : a.M - 1;
        sSx[r * ng + g] = a.sx[(size_t)t * ng + g];
    }
    for (int i = tid; i < BN * ng; i += NT) {
        const int r = i / ng, g = i - r * ng;
        sSw[r * ng + g] = a.sw[(size_t)(n0 + r) * ng + g];
    }
    __syncthreads();

    v16i acc[2][JT];
    float facc[2][JT][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) { acc[i][j][r] = 0; facc[i][j][r] = 0.0f; }

    // operand rows of this lane: A row (token) wm*64 + 32 i + lane % 32, B row (weight row)
    // wn*BN/2 + 32 j + lane % 32; both take chunk 2 kk + lane / 32 of the stage's 32-byte K slice
    // kk, so A and B pair the same K positions
    const int arow = wm * 64 + (lane & 31), brow = wn * (BN / 2) + (lane & 31);
    const int swa = (arow >> 2) & 3, swb = (brow >> 2) & 3, kh = lane >> 5;
    for (int s = 0; s < nsteps; ++s) {
        // this wave's transfers for stage s are done once at most the NI (kGS - 2) issued after
        // them are outstanding (vector-memory counts retire in order); after the barrier every
        // wave's are, and every wave has finished reading stage s - 1, whose slot is refilled now
        // with stage s + kGS - 1 (past the end: stage 0 again, never read, so every iteration
        // issues the same transfers and the count stays exact)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(NI * (kGS - 2)));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        __builtin_amdgcn_sched_barrier(0);
        const int sn = s + kGS - 1;
        issue(sn < nsteps ? sn : 0, sn % kGS);
        const int8_t* st = sR + (s % kGS) * kGStage;
#pragma unroll
        for (int kk = 0; kk < kGK / 32; ++kk) {
            const int c = 2 * kk + kh;
            v4i av[2], bv[JT];
#pragma unroll
            for (int i = 0; i < 2; ++i) av[i] = *(const v4i*)(st + (arow + 32 * i) * kGK + ((c ^ swa) << 4));
#pragma unroll
            for (int j = 0; j < JT; ++j) bv[j] = *(const v4i*)(st + (kGM + brow + 32 * j) * kGK + ((c ^ swb) << 4));
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < JT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if ((s + 1) % spg == 0) {
            // fold the group: accumulator element r of a 32 x 32 tile is row
            // 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32
            const int g = (s + 1) / spg - 1;
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                const float swv = sSw[(brow + 32 * j) * ng + g];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int tr = wm * 64 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                        const float sc = swv * sSx[tr * ng + g];
                        facc[i][j][r] = __builtin_fmaf((float)acc[i][j][r], sc, facc[i][j][r]);
                        acc[i][j][r] = 0;
                    }
            }
        }
    }
    // no transfer may still be writing LDS when the block ends
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            const int n = n0 + wn * (BN / 2) + 32 * j + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int t = m0 + wm * 64 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (t < a.M) {
                    float o = facc[i][j][r] * alpha_of(a.alpha, a.asel, n);
                    if (a.res) o = o + a.rs * (a.res_bf16 ? bf2f(((const uint16_t*)a.res)[(size_t)t * a.ldr + n])
                                                          : a.res[(size_t)t * a.ldr + n]);
                    if (a.out_bf16) ((uint16_t*)a.y)[(size_t)t * a.ldy + n] = f2bf(o);
                    else a.y[(size_t)t * a.ldy + n] = o;
                }
            }
        }
}

// The same GEMM for 256-token tiles with register-staged loads and 128-byte stages: each thread
// moves six 16-byte chunks per stage with plain vector loads, issued three stages ahead into two
// register sets, and writes them to a double-buffered LDS stage one iteration before the
// multiply; 16 MFMAs per wave between barriers, each 32-byte slice's operands read from LDS
// while the previous slice multiplies. The loop is unrolled by two so the register sets
// are named at compile time; nsteps (K / 128) must be even. Rows are 128 bytes, chunk c of row R
// in slot c ^ ((R >> 1) & 7) (the 16 rows one operand read serves fill a 256-byte bank window).
// Same fold and tile order as k_gemm_i8g.
template <int RES, bool OBF>   // epilogue form, as k_gemm_i8g_w4's
__global__ __launch_bounds__(512) void k_gemm_i8g_rs(GemmArgs a) {
    constexpr int BM = 256, BN = kGN, NT = 512, KB = 128, kStage = (BM + BN) * KB;
    __shared__ __align__(16) int8_t sR[2 * kStage];
    extern __shared__ float sScl[];
    float* sSx = sScl;
    float* sSw = sScl + BM * a.ng;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int nt = a.N / BN, mt = (a.M + BM - 1) / BM, T = nt * mt;
    const int b = blockIdx.x;
    const int tile = (T % 8 == 0) ? (b % 8) * (T / 8) + b / 8 : b;
    const int grp = tile / (4 * nt), fm = grp * 4, gsz = (mt - fm < 4) ? mt - fm : 4;
    const int within = tile - grp * 4 * nt;
    const int m0 = (fm + within % gsz) * BM, n0 = (within / gsz) * BN;
    const int K = a.K, ng = a.ng, spg = a.gs / KB, nsteps = K / KB;

    // thread tid moves chunk q = tid + 512 k (k < 6) of each stage: stage row q / 8 (A rows
    // first), natural chunk q % 8 of that row, stored at slot (q % 8) ^ ((row >> 1) & 7)
    const int8_t* gp[6];
    int lo[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int q = tid + NT * k, rs = q >> 3, c = q & 7;
        const int r = rs < BM ? rs : rs - BM;
        if (rs < BM) {
            const int t = (m0 + r < a.M) ? m0 + r : a.M - 1;
            gp[k] = a.x + (size_t)t * K + 16 * c;
        } else {
            gp[k] = a.w + (size_t)(n0 + r) * K + 16 * c;
        }
        lo[k] = rs * KB + ((c ^ ((r >> 1) & 7)) << 4);
    }
    uint4 ra0, ra1, ra2, ra3, ra4, ra5, rb0, rb1, rb2, rb3, rb4, rb5;
#define Q27X_LD(R0, R1, R2, R3, R4, R5, step)                                                       \
    { const int k0_ = (step) * KB;                                                                  \
      R0 = *(const uint4*)(gp[0] + k0_); R1 = *(const uint4*)(gp[1] + k0_);                         \
      R2 = *(const uint4*)(gp[2] + k0_); R3 = *(const uint4*)(gp[3] + k0_);                         \
      R4 = *(const uint4*)(gp[4] + k0_); R5 = *(const uint4*)(gp[5] + k0_); }
#define Q27X_ST(R0, R1, R2, R3, R4, R5, slot)                                                       \
    { int8_t* d_ = sR + (slot) * kStage;                                                            \
      *(uint4*)(d_ + lo[0]) = R0; *(uint4*)(d_ + lo[1]) = R1; *(uint4*)(d_ + lo[2]) = R2;           \
      *(uint4*)(d_ + lo[3]) = R3; *(uint4*)(d_ + lo[4]) = R4; *(uint4*)(d_ + lo[5]) = R5; }

    for (int i = tid; i < BM * ng; i += NT) {
        const int r = i / ng, g = i - r * ng;
        const int t = (m0 + r < a.M) ? m0 + r : a.M - 1;
        sSx[r * ng + g] = a.sx[(size_t)t * ng + g];
    }
    for (int i = tid; i < BN * ng; i += NT) {
        const int r = i / ng, g = i - r * ng;
        sSw[r * ng + g] = a.sw[(size_t)(n0 + r) * ng + g];
    }
    // stages 0 and 1 in flight, stage 0 to LDS, stage 2 in flight behind stage 1
    Q27X_LD(ra0, ra1, ra2, ra3, ra4, ra5, 0)
    Q27X_LD(rb0, rb1, rb2, rb3, rb4, rb5, 1)
    Q27X_ST(ra0, ra1, ra2, ra3, ra4, ra5, 0)
    Q27X_LD(ra0, ra1, ra2, ra3, ra4, ra5, 2 < nsteps ? 2 : 0)
    __syncthreads();

    v16i acc[2][2];
    float facc[2][2][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) { acc[i][j][r] = 0; facc[i][j][r] = 0.0f; }
    const int arow = wm * 64 + (lane & 31), brow = wn * 64 + (lane & 31);
    const int swa = (arow >> 1) & 7, swb = (brow >> 1) & 7, kh = lane >> 5;

    // iteration s: multiply stage s (LDS slot s % 2); store stage s + 1 (register set (s + 1) % 2)
    // into the other slot; reload that set with stage s + 3 (past the end: stage 0, stored into a
    // slot nobody reads again); barrier
#define Q27X_ITER(S_, N0, N1, N2, N3, N4, N5)                                                       \
    {                                                                                               \
        const int s_ = (S_);                                                                        \
        const int8_t* st = sR + (s_ & 1) * kStage;                                                  \
        v4i av[2][2], bv[2][2];                                                                     \
_Pragma("unroll")                                                                                   \
        for (int i = 0; i < 2; ++i) av[0][i] = *(const v4i*)(st + (arow + 32 * i) * KB + ((kh ^ swa) << 4)); \
_Pragma("unroll")                                                                                   \
        for (int j = 0; j < 2; ++j) bv[0][j] = *(const v4i*)(st + (BM + brow + 32 * j) * KB + ((kh ^ swb) << 4)); \
_Pragma("unroll")                                                                                   \
        for (int kk = 0; kk < KB / 32; ++kk) {                                                      \
            const int cu = kk & 1, nx = cu ^ 1;                                                     \
            if (kk + 1 < KB / 32) {                                                                 \
                const int c = 2 * (kk + 1) + kh;                                                    \
_Pragma("unroll")                                                                                   \
                for (int i = 0; i < 2; ++i) av[nx][i] = *(const v4i*)(st + (arow + 32 * i) * KB + ((c ^ swa) << 4)); \
_Pragma("unroll")                                                                                   \
                for (int j = 0; j < 2; ++j) bv[nx][j] = *(const v4i*)(st + (BM + brow + 32 * j) * KB + ((c ^ swb) << 4)); \
            }                                                                                       \
_Pragma("unroll")                                                                                   \
            for (int i = 0; i < 2; ++i)                                                             \
_Pragma("unroll")                                                                                   \
                for (int j = 0; j < 2; ++j)                                                         \
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[cu][i], bv[cu][j], acc[i][j], 0, 0, 0); \
        }                                                                                           \
        if ((s_ + 1) % spg == 0) {                                                                  \
            const int g = (s_ + 1) / spg - 1;                                                       \
_Pragma("unroll")                                                                                   \
            for (int j = 0; j < 2; ++j) {                                                           \
                const float swv = sSw[(brow + 32 * j) * ng + g];                                    \
_Pragma("unroll")                                                                                   \
                for (int i = 0; i < 2; ++i)                                                         \
_Pragma("unroll")                                                                                   \
                    for (int r = 0; r < 16; ++r) {                                                  \
                        const int tr = wm * 64 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); \
                        const float sc = swv * sSx[tr * ng + g];                                    \
                        facc[i][j][r] = __builtin_fmaf((float)acc[i][j][r], sc, facc[i][j][r]);     \
                        acc[i][j][r] = 0;                                                           \
                    }                                                                               \
            }                                                                                       \
        }                                                                                           \
        Q27X_ST(N0, N1, N2, N3, N4, N5, (s_ + 1) & 1)                                               \
        Q27X_LD(N0, N1, N2, N3, N4, N5, s_ + 3 < nsteps ? s_ + 3 : 0)                               \
        __syncthreads();                                                                            \
    }
    for (int s = 0; s < nsteps; s += 2) {
        Q27X_ITER(s, rb0, rb1, rb2, rb3, rb4, rb5)        // stage s + 1 sits in the b set
        Q27X_ITER(s + 1, ra0, ra1, ra2, ra3, ra4, ra5)    // stage s + 2 in the a set
    }
#undef Q27X_ITER
#undef Q27X_LD
#undef Q27X_ST

    // outputs (32-bit element offsets: the launcher keeps M x ldy and M x ldr below 2^30)
    const uint32_t nb = (uint32_t)(n0 + wn * 64 + (lane & 31));
    float al[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) al[j] = alpha_of(a.alpha, a.asel, (int)nb + 32 * j);
    auto out = [&](auto full) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int t = m0 + wm * 64 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (decltype(full)::value || t < a.M) {
                    const uint32_t yo = (uint32_t)t * (uint32_t)a.ldy + nb;
                    const uint32_t ro = (uint32_t)t * (uint32_t)a.ldr + nb;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        float o = facc[i][j][r] * al[j];
                        if constexpr (RES == 1) o = o + a.rs * a.res[ro + 32 * j];
                        if constexpr (RES == 2) o = o + a.rs * bf2f(((const uint16_t*)a.res)[ro + 32 * j]);
                        if constexpr (OBF) ((uint16_t*)a.y)[yo + 32 * j] = f2bf(o);
                        else a.y[yo + 32 * j] = o;
                    }
                }
            }
    };
    if (m0 + BM <= a.M) out(std::true_type{});
    else out(std::false_type{});
}

// One group over the whole K (the reference's default arm) on 256-token x 256-row tiles: 8 waves,
// two per SIMD, each owning 128 tokens x 64 rows as 4 x 2 v_mfma_i32_32x32x32_i8 tiles (128
// accumulator registers; no fp32 group accumulators are needed, the scales apply once at the end),
// so each MFMA reads three quarters of a KiB of LDS operands instead of the 64 x 64 quarter's full
// KiB, and while one wave of a SIMD waits (a barrier, its operand reads) the other multiplies
// (with 4 waves of 128 x 128, one per SIMD, the same tile ran 17-20% slower). K
// advances 128 bytes per stage (each stage row is one whole 128-byte line of a row, which halves
// the load requests of 64-byte stages) through two 64 KiB LDS stages filled by LDS DMA. The
// operand reads are pipelined one 32-byte slice ahead of the MFMAs, across the stage barrier too:
// the barrier that certifies stage s + 1 sits before the last slice of stage s, whose operands
// are already in registers, and the next stage's first slice is read while that slice multiplies.
// Rows are 128 bytes, chunk c of row R in slot c ^ ((R >> 1) & 7) (the 16 rows of one operand read
// fill a 256-byte bank window). Same tile order as k_gemm_i8g; the int32 sums are exact, so the
// outputs are the other kernels' bits.
constexpr int kW4B = 256, kW4K = 128, kW4S = 2;
constexpr int kW4Stage = 2 * kW4B * kW4K;              // 64 KiB: A rows, then B rows
constexpr int kW4NI = kW4Stage / (1024 * 8);           // 1 KiB transfers per wave per stage (8)
// RES: no residual (0), fp32 (1) or bf16 (2) residual rows; OBF: bf16 output. Instances per
// epilogue form: with per-element branches on them the unrolled epilogue of 256 values per lane
// cost ~20 us per tile.
template <int RES, bool OBF>
__global__ __launch_bounds__(512) void k_gemm_i8g_w4(GemmArgs a) {
    __shared__ __align__(16) int8_t sR[kW4S * kW4Stage];
    __shared__ float sSx[kW4B], sSw[kW4B];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    const int nt = a.N / kW4B, mt = (a.M + kW4B - 1) / kW4B, T = nt * mt;
    const int b = blockIdx.x;
    const int tile = (T % 8 == 0) ? (b % 8) * (T / 8) + b / 8 : b;
    const int grp = tile / (4 * nt), fm = grp * 4, gsz = (mt - fm < 4) ? mt - fm : 4;
    const int within = tile - grp * 4 * nt;
    const int m0 = (fm + within % gsz) * kW4B, n0 = (within / gsz) * kW4B;
    const int K = a.K, nsteps = K / kW4K;
    // DMA: transfer i (< 8) of wave w fills stage rows 8 (8 w + i) .. +8; lane l writes row
    // 8 (8 w + i) + l / 8, slot l % 8, so it loads that row's chunk (l % 8) ^ ((row >> 1) & 7)
    // (waves 0-3 fill the A rows, waves 4-7 the B rows: one base per wave, byte offsets below
    // 2^31 for the row counts and K this kernel takes)
    const int8_t* gb = wave < 4 ? a.x : a.w;
    uint32_t go[kW4NI];
#pragma unroll
    for (int i = 0; i < kW4NI; ++i) {
        const int rs = 8 * (kW4NI * wave + i) + (lane >> 3);
        const int r = rs < kW4B ? rs : rs - kW4B;
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int row = rs < kW4B ? ((m0 + r < a.M) ? m0 + r : a.M - 1) : n0 + r;   // rows past M repeat row M - 1
        go[i] = (uint32_t)row * (uint32_t)K + 16 * c;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sR;
    auto issue = [&](int step, int slot) __attribute__((always_inline)) {
        const uint32_t base = lds0 + slot * kW4Stage + 1024 * kW4NI * wave;
#pragma unroll
        for (int i = 0; i < kW4NI; ++i)
            lds_dma16(gb + go[i] + (uint32_t)(step * kW4K), __builtin_amdgcn_readfirstlane(base + 1024 * i));
    };
    issue(0, 0);
    if (tid < kW4B) {
        const int t = (m0 + tid < a.M) ? m0 + tid : a.M - 1;
        sSx[tid] = a.sx[t];
        sSw[tid] = a.sw[n0 + tid];
    }
    v16i acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    // operand rows of this lane: A (token) wm*128 + 32 i + lane % 32, B (weight row) wn*64 + 32 j +
    // lane % 32; both take chunk 2 kk + lane / 32 of the stage's 32-byte K slice kk
    const int arow = wm * 128 + (lane & 31), brow = kW4B + wn * 64 + (lane & 31);
    const int swa = (arow >> 1) & 7, swb = ((brow - kW4B) >> 1) & 7, kh = lane >> 5;
    auto rd = [&](v4i (&av)[4], v4i (&bv)[2], int slot, int kk) __attribute__((always_inline)) {
        const int8_t* st = sR + slot * kW4Stage;
        const int c = 2 * kk + kh;
#pragma unroll
        for (int i = 0; i < 4; ++i) av[i] = *(const v4i*)(st + (arow + 32 * i) * kW4K + ((c ^ swa) << 4));
#pragma unroll
        for (int j = 0; j < 2; ++j) bv[j] = *(const v4i*)(st + (brow + 32 * j) * kW4K + ((c ^ swb) << 4));
    };
    auto mm = [&](const v4i (&av)[4], const v4i (&bv)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[i], bv[j], acc[i][j], 0, 0, 0);
    };
    // this wave's transfers of the next stage done and its operand reads of the current one
    // returned; after the barrier every wave's are (nothing is scheduled across it)
    auto sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0) & ~(15 << 8));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int SL = kW4K / 32;                      // 32-byte slices per stage
    v4i oa[2][4], ob[2][2];
    sync();                                            // stage 0 everywhere (and the scales)
    issue(1 < nsteps ? 1 : 0, 1);
    rd(oa[0], ob[0], 0, 0);
    for (int s = 0; s < nsteps; ++s) {
#pragma unroll
        for (int kk = 0; kk < SL; ++kk) {
            const int cu = kk & 1, nx = cu ^ 1;
            if (kk + 1 < SL) {
                rd(oa[nx], ob[nx], s & 1, kk + 1);
            } else {
                // stage s + 1 landed everywhere and stage s is read by all: its slot takes stage
                // s + 2 (past the end: stage 0 again into a slot nobody reads, so every iteration
                // issues the same transfers); the next stage's first slice is read meanwhile
                // (past the last stage that is a stale slot, not used)
                sync();
                issue(s + 2 < nsteps ? s + 2 : 0, s & 1);
                rd(oa[nx], ob[nx], (s + 1) & 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
            mm(oa[cu], ob[cu]);
            __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
        }
    }
    // no transfer may still be writing LDS when the block ends
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    // the tile's outputs; rows past M only in the last token tile. Element offsets are 32-bit
    // (the launcher keeps M x ldy and M x ldr below 2^30), so the stores take the output's base in
    // scalar registers.
    const uint32_t nb = (uint32_t)(n0 + wn * 64 + (lane & 31));
    float swv[2], al[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        swv[j] = sSw[wn * 64 + 32 * j + (lane & 31)];
        al[j] = alpha_of(a.alpha, a.asel, (int)nb + 32 * j);
    }
    auto out = [&](auto full) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int tl = wm * 128 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), t = m0 + tl;
                if (decltype(full)::value || t < a.M) {
                    const float sxv = sSx[tl];
                    const uint32_t yo = (uint32_t)t * (uint32_t)a.ldy + nb;
                    const uint32_t ro = (uint32_t)t * (uint32_t)a.ldr + nb;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        float o = __builtin_fmaf((float)acc[i][j][r], swv[j] * sxv, 0.0f) * al[j];
                        if constexpr (RES == 1) o = o + a.rs * a.res[ro + 32 * j];
                        if constexpr (RES == 2) o = o + a.rs * bf2f(((const uint16_t*)a.res)[ro + 32 * j]);
                        if constexpr (OBF) ((uint16_t*)a.y)[yo + 32 * j] = f2bf(o);
                        else a.y[yo + 32 * j] = o;
                    }
                }
            }
    };
    if (m0 + kW4B <= a.M) out(std::true_type{});
    else out(std::false_type{});
}

// 128-byte stages (a stage row is one whole 128-byte line of a row) through a ring of S LDS stages filled by LDS
// DMA: 64 WM tokens x 64 WN weight rows per block, each wave 64 x 64 as 2 x 2 v_mfma_i32_32x32x32_i8 tiles; with
// KS = 2 two waves share a 64 x 64 quarter, each multiplying two of the stage's four 32-byte slices (their sums meet
// in LDS at the end). Operand reads run one slice ahead of the MFMAs, across the stage barrier too, as in
// k_gemm_i8g_w4. Same tile order and row swizzle.
template <int WM, int WN, int KS, int S> struct RingCfg {
    static constexpr int BM = 64 * WM, BN = 64 * WN, NW = WM * WN * KS;
    static constexpr int Stage = (BM + BN) * 128, NI = Stage / (1024 * NW);
    static constexpr int Ring = S * Stage;
    static_assert(Stage % (1024 * NW) == 0 && NI * (S - 1) < 64, "whole transfers per wave");
};
template <int WM, int WN, int KS, int S, bool GRP>
__global__ __launch_bounds__(64 * WM * WN * KS) void k_gemm_i8g_ring(GemmArgs a) {
    using C = RingCfg<WM, WN, KS, S>;
    static_assert(!GRP || KS == 1, "group sums are folded by one wave");
    constexpr int BM = C::BM, BN = C::BN, NT = 64 * C::NW, NI = C::NI, SL = 4 / KS;
    extern __shared__ __attribute__((aligned(16))) int8_t rgdyn[];     // [S][Stage] | scales [BM][ng] | [BN][ng]
    float* sSx = (float*)(rgdyn + C::Ring);
    float* sSw = sSx + BM * a.ng;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
    const int nt = a.N / BN, mt = (a.M + BM - 1) / BM, T = nt * mt;
    const int b = blockIdx.x, xq = T / 8, xr = T % 8, xi = b % 8;
    const int tile = xi * xq + (xi < xr ? xi : xr) + b / 8;
    const int grp = tile / (4 * nt), fm = grp * 4, gsz = (mt - fm < 4) ? mt - fm : 4;
    const int within = tile - grp * 4 * nt;
    const int m0 = (fm + within % gsz) * BM, n0 = (within / gsz) * BN;
    const int K = a.K, ng = a.ng, nst = K / 128, spg = a.gs / 128;
    uint32_t off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int rs = 8 * (NI * wave + i) + (lane >> 3), r = rs < BM ? rs : rs - BM;
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        off[i] = (uint32_t)(rs >= BM ? n0 + r : m0 + r < a.M ? m0 + r : a.M - 1) * (uint32_t)K + 16u * c;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)rgdyn + 1024 * NI * wave;
    auto issue = [&](int st, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
            lds_dma16_at((8 * (NI * wave + i) < BM ? a.x : a.w) + (size_t)st * 128, off[i],
                         __builtin_amdgcn_readfirstlane(lds0 + slot * C::Stage + 1024 * i));
    };
#pragma unroll
    for (int p = 0; p < S; ++p) issue(p < nst ? p : 0, p);
    for (int i = tid; i < BM * ng; i += NT) {
        const int r = i / ng, t = m0 + r < a.M ? m0 + r : a.M - 1;
        sSx[i] = a.sx[(size_t)t * ng + (i - r * ng)];
    }
    for (int i = tid; i < BN * ng; i += NT) sSw[i] = a.sw[(size_t)n0 * ng + i];
    v16i acc[2][2];
    float facc[GRP ? 2 : 1][GRP ? 2 : 1][GRP ? 16 : 1];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0;
                if constexpr (GRP) facc[i][j][r] = 0.0f;
            }
    const int arow = wm * 64 + (lane & 31), brow = wn * 64 + (lane & 31);
    const int swa = (arow >> 1) & 7, swb = (brow >> 1) & 7, kh = lane >> 5;
    auto rd = [&](v4i (&av)[2], v4i (&bv)[2], int slot, int kk) __attribute__((always_inline)) {
        const int8_t* st = rgdyn + slot * C::Stage;
        const int c = 2 * (SL * kg + kk) + kh;
#pragma unroll
        for (int i = 0; i < 2; ++i) av[i] = *(const v4i*)(st + (arow + 32 * i) * 128 + ((c ^ swa) << 4));
#pragma unroll
        for (int j = 0; j < 2; ++j) bv[j] = *(const v4i*)(st + (BM + brow + 32 * j) * 128 + ((c ^ swb) << 4));
    };
    // at most `left` stages' transfers of this wave outstanding and its operand reads returned, then the barrier
    auto sync = [&](auto left) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(NI * decltype(left)::value) & ~(15 << 8));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        __builtin_amdgcn_sched_barrier(0);
    };
    v4i oa[2][2], ob[2][2];
    sync(std::integral_constant<int, S - 1>{});
    rd(oa[0], ob[0], 0, 0);
    int slot = 0, gl = spg, g = 0;
    for (int s = 0; s < nst; ++s) {
        const int sn = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
        for (int kk = 0; kk < SL; ++kk) {
            const int cu = kk & 1, nx = cu ^ 1;
            if (kk + 1 < SL) {
                rd(oa[nx], ob[nx], slot, kk + 1);
            } else {
                // stage s + 1 landed everywhere and stage s is read by all: its slot takes stage s + S (past the
                // end: stage 0 again, so every iteration issues the same transfers)
                sync(std::integral_constant<int, S - 2>{});
                issue(s + S < nst ? s + S : 0, slot);
                rd(oa[nx], ob[nx], sn, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(oa[cu][i], ob[cu][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        }
        slot = sn;
        if constexpr (GRP) {
            if (--gl == 0) {
                gl = spg;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float swv = sSw[(brow + 32 * j) * ng + g];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int tr = wm * 64 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                            facc[i][j][r] = __builtin_fmaf((float)acc[i][j][r], swv * sSx[tr * ng + g], facc[i][j][r]);
                            acc[i][j][r] = 0;
                        }
                }
                ++g;
            }
        }
    }
    // no transfer may still be writing LDS when the block ends
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    if constexpr (KS == 2) {
        // the two slice halves of a quarter: each wave gives the other its sums of the other's token half
        __syncthreads();
        int* ex = (int*)rgdyn + (wave % (WM * WN)) * 2 * 32 * 64 + lane;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) ex[((kg ^ 1) * 32 + j * 16 + r) * 64] = kg ? acc[0][j][r] : acc[1][j][r];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][j][r] = (kg ? acc[1][j][r] : acc[0][j][r]) + ex[(kg * 32 + j * 16 + r) * 64];
    }
    const uint32_t nb = (uint32_t)(n0 + wn * 64 + (lane & 31));
    float swv[2], al[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        swv[j] = GRP ? 0.0f : sSw[wn * 64 + 32 * j + (lane & 31)];
        al[j] = alpha_of(a.alpha, a.asel, (int)nb + 32 * j);
    }
    auto out = [&](auto res, auto obf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2 / KS; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int tl = wm * 64 + 32 * (KS == 2 ? kg : i) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), t = m0 + tl;
                if (t < a.M) {
                    const uint32_t yo = (uint32_t)t * (uint32_t)a.ldy + nb, ro = (uint32_t)t * (uint32_t)a.ldr + nb;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        float o;
                        if constexpr (GRP) o = facc[i][j][r] * al[j];
                        else o = __builtin_fmaf((float)acc[i][j][r], swv[j] * sSx[tl], 0.0f) * al[j];
                        if constexpr (decltype(res)::value == 1) o = o + a.rs * a.res[ro + 32 * j];
                        if constexpr (decltype(res)::value == 2) o = o + a.rs * bf2f(((const uint16_t*)a.res)[ro + 32 * j]);
                        if constexpr (decltype(obf)::value) ((uint16_t*)a.y)[yo + 32 * j] = f2bf(o);
                        else a.y[yo + 32 * j] = o;
                    }
                }
            }
    };
    auto form = [&](auto res) __attribute__((always_inline)) {
        if (a.out_bf16) out(res, std::true_type{});
        else out(res, std::false_type{});
    };
    if (!a.res) form(std::integral_constant<int, 0>{});
    else if (a.res_bf16) form(std::integral_constant<int, 2>{});
    else form(std::integral_constant<int, 1>{});
}

// Few tokens, or few weight rows for the CUs: a block of NW waves owns 16 RT weight rows x 16 MT tokens and its
// waves split K, so every wave keeps the whole tile in registers (RT x MT v_mfma_i32_16x16x64_i8 tiles) and moves
// its own operands through its own LDS ring (S stages of 128 K bytes, LDS DMA): the main loop has no barrier. The
// waves' int32 sums are exact in any order: they meet in LDS (ds_add) in one slot per group, then every thread
// folds its outputs in group order. gpp groups fit the slots at a time; more groups take further phases, whose
// transfers are already in flight.
template <int RT, int MT, int NW, int S> struct SkCfg {
    static constexpr int Rows = 16 * (RT + MT), Stage = Rows * 128, NI = Rows / 8;    // 1 KiB transfers per stage
    static constexpr int Ring = NW * S * Stage;
    static constexpr int Out = 256 * RT * MT;          // outputs of the tile
    static_assert(NI * (S - 1) < 64, "vector-memory count");
};
template <int RT, int MT, int NW, int S>
__global__ __launch_bounds__(64 * NW) void k_gemm_i8g_sk(GemmArgs a, int gpp) {
    using C = SkCfg<RT, MT, NW, S>;
    constexpr int NT = 64 * NW, NO = C::Out, NPT = (NO + NT - 1) / NT, NI = C::NI;
    // rings [NW][S][Stage] | [gpp][NO] int32 | token scales [16 MT][ng] | row scales [16 RT][ng]
    extern __shared__ __attribute__((aligned(16))) int8_t skdyn[];
    const int ng = a.ng, K = a.K;
    int* sAcc = (int*)(skdyn + C::Ring);
    float* sSx = (float*)(sAcc + (size_t)gpp * NO);
    float* sSw = sSx + 16 * MT * ng;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // tiles with the token tile fastest, in one contiguous run per XCD (blocks go to the XCDs round-robin), so the
    // blocks that share weight rows share an L2
    const int mt = (a.M + 16 * MT - 1) / (16 * MT), T = gridDim.x, b = blockIdx.x;
    const int xq = T / 8, xr = T % 8, xi = b % 8;
    const int tile = xi * xq + (xi < xr ? xi : xr) + b / 8;
    const int m0 = (tile % mt) * 16 * MT, n0 = (tile / mt) * 16 * RT;
    // transfer i fills stage rows 8 i .. 8 i + 7 (weight rows, then tokens): lane l row 8 i + l / 8, slot l % 8, which
    // holds chunk (l % 8) ^ ((row >> 1) & 7) of the row's 128 bytes (rows past M repeat row M - 1)
    uint32_t off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int row = 8 * i + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        const int t = m0 + row - 16 * RT;
        off[i] = (uint32_t)(i < 2 * RT ? n0 + row : t < a.M ? t : a.M - 1) * (uint32_t)K + 16u * c;
    }
    const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)skdyn + wave * S * C::Stage;
    auto issue = [&](int st, int slot) __attribute__((always_inline)) {
        const int8_t* px = a.x + (size_t)st * 128;
        const int8_t* pw = a.w + (size_t)st * 128;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            lds_dma16_at(i < 2 * RT ? pw : px, off[i], __builtin_amdgcn_readfirstlane(ring + slot * C::Stage + 1024 * i));
    };
    const int nst = K / 128, spg = a.gs / 128, spp = spg * gpp;      // stages: all, per group, per phase
    // this wave's stages of the phase that starts at stage p0
    auto range = [&](int p0, int& s0, int& s1) __attribute__((always_inline)) {
        const int pn = nst - p0 < spp ? nst - p0 : spp;
        s0 = p0 + pn * wave / NW;
        s1 = p0 + pn * (wave + 1) / NW;
    };
    // the stage to issue next: the wave's ranges one after another (past the last: stage 0 again, so every iteration
    // issues the same transfers and the count stays exact)
    int ip = 0, is = 0, ie = 0;
    range(0, is, ie);
    auto next = [&]() __attribute__((always_inline)) {
        while (is >= ie && ip + spp < nst) { ip += spp; range(ip, is, ie); }
        return is < ie ? is++ : 0;
    };
#pragma unroll
    for (int p = 0; p < S - 1; ++p) issue(next(), p);
    for (int i = tid; i < 16 * MT * ng; i += NT) {
        const int r = i / ng, t = m0 + r < a.M ? m0 + r : a.M - 1;
        sSx[i] = a.sx[(size_t)t * ng + (i - r * ng)];
    }
    for (int i = tid; i < 16 * RT * ng; i += NT) sSw[i] = a.sw[(size_t)n0 * ng + i];
    for (int i = tid; i < gpp * NO; i += NT) sAcc[i] = 0;
    __syncthreads();
    v4i acc[RT][MT];
    float o[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) o[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = v4i{0, 0, 0, 0};
    const int sw = (lane & 15) >> 1;                   // ((row >> 1) & 7) of this lane's operand rows
    int slot = 0;
    for (int p0 = 0, g0 = 0; p0 < nst; p0 += spp, g0 += gpp) {
        const int gn = (nst - p0 < spp ? nst - p0 : spp) / spg;
        int s0, s1;
        range(p0, s0, s1);
        int left = spg - s0 % spg, as = s0 / spg - g0;               // stages left of the current group, its slot
        for (int s = s0; s < s1; ++s) {
            // the slot read in the iteration before takes the stage S - 1 ahead; this stage has landed once at
            // most the S - 1 stages behind it are outstanding (vector-memory counts retire in order)
            issue(next(), slot == 0 ? S - 1 : slot - 1);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(NI * (S - 1)));
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            __builtin_amdgcn_sched_barrier(0);
            const int8_t* st = skdyn + (wave * S + slot) * C::Stage + (lane & 15) * 128;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const int c = ((4 * kk + (lane >> 4)) ^ sw) << 4;
                v4i wv[RT], xv[MT];
#pragma unroll
                for (int j = 0; j < RT; ++j) wv[j] = *(const v4i*)(st + 16 * j * 128 + c);
#pragma unroll
                for (int i = 0; i < MT; ++i) xv[i] = *(const v4i*)(st + 16 * (RT + i) * 128 + c);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < RT; ++j)
                        acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv[i], wv[j], acc[j][i], 0, 0, 0);
            }
            slot = slot + 1 == S ? 0 : slot + 1;
            if (--left == 0 || s + 1 == s1) {
#pragma unroll
                for (int j = 0; j < RT; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            __hip_atomic_fetch_add(&sAcc[as * NO + ((j * MT + i) * 4 + r) * 64 + lane], acc[j][i][r],
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            acc[j][i][r] = 0;
                        }
                ++as;
                left = spg;
            }
            // (the operand reads above have returned: their values are consumed before the slot is refilled)
            __builtin_amdgcn_s_waitcnt(0xC07F);         // lgkmcnt(0)
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        // output u: element r of lane's result in tile (j, i): token 16 i + 4 (lane / 16) + r, row 16 j + lane % 16
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int u = tid + NT * i;
            if (u < NO) {
                const int tl = u >> 8, r = (u >> 6) & 3;
                const float* px = sSx + (16 * (tl % MT) + 4 * (lane >> 4) + r) * ng + g0;
                const float* pw = sSw + (16 * (tl / MT) + (lane & 15)) * ng + g0;
                for (int g = 0; g < gn; ++g) {
                    o[i] = __builtin_fmaf((float)sAcc[g * NO + u], pw[g] * px[g], o[i]);
                    sAcc[g * NO + u] = 0;
                }
            }
        }
        if (p0 + spp < nst) __syncthreads();                        // the slots are read and cleared
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));          // no transfer may still be writing LDS when the block ends
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const int u = tid + NT * i, tl = u >> 8, r = (u >> 6) & 3;
        const int t = m0 + 16 * (tl % MT) + 4 * (lane >> 4) + r, n = n0 + 16 * (tl / MT) + (lane & 15);
        if (u < NO && t < a.M) {
            float v = o[i] * alpha_of(a.alpha, a.asel, n);
            if (a.res) v = v + a.rs * (a.res_bf16 ? bf2f(((const uint16_t*)a.res)[(size_t)t * a.ldr + n])
                                                  : a.res[(size_t)t * a.ldr + n]);
            if (a.out_bf16) ((uint16_t*)a.y)[(size_t)t * a.ldy + n] = f2bf(v);
            else a.y[(size_t)t * a.ldy + n] = v;
        }
    }
}

// Weights: per-64 mirror -> per-(row, group) codes and scales; one wave per (row, group). In place when wg == w (each
// element is read and written by the same thread). Bound by memory: 16 codes per lane and load, four loads in flight
// (a byte per lane and load: 16384 x 5120 96 us, now 34: 4.9 TB/s). A pass is 4096 codes whatever the group, so with
// narrower groups lanes load and convert codes that they do not store: on cached codes, in groups of 5120 68 us and now
// 28, of 1024 87 / 31, of 256 155 / 104, of 64 494 / 408. VEC = 0 is the byte form, for codes that are not 16-byte aligned.
template <bool VEC>
__global__ __launch_bounds__(256) void k_i8g64_to_grp(const int8_t* w, const float* s64, int rows, int K, int gs,
                                                      int8_t* wg, float* sg) {
    const int ng = K / gs, lane = threadIdx.x & 63;
    const long long u = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (u >= (long long)rows * ng) return;
    const int8_t* src = w + (size_t)u * gs;
    int8_t* dst = wg + (size_t)u * gs;
    const float* sr = s64 + (size_t)u * (gs >> 6);
    float mx = 0.0f;
    for (int i = lane; i < (gs >> 6); i += 64) mx = fmaxf(mx, sr[i]);
    if constexpr (VEC) {
        constexpr int U = 4;
        uint4 c[U];
        float sc[U];
        auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int k = k0 + 1024 * i + 16 * lane, kc = k < gs ? k : 0;
                c[i] = *(const uint4*)(src + kc);
                sc[i] = sr[kc >> 6];
            }
        };
        load(0);
        mx = max_xor(mx, 64);
        const float inv = (mx > 0.0f) ? 1.0f / mx : 0.0f;
        if (lane == 0) sg[u] = mx;
        for (int k0 = 0; k0 < gs; k0 += 1024 * U) {
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int k = k0 + 1024 * i + 16 * lane;
                const uint32_t in[4] = {c[i].x, c[i].y, c[i].z, c[i].w};
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = pack4(qcode((float)(int8_t)in[e] * sc[i], inv), qcode((float)(int8_t)(in[e] >> 8) * sc[i], inv),
                                 qcode((float)(int8_t)(in[e] >> 16) * sc[i], inv), qcode((float)(int8_t)(in[e] >> 24) * sc[i], inv));
                if (k < gs) *(uint4*)(dst + k) = make_uint4(o[0], o[1], o[2], o[3]);
            }
            if (k0 + 1024 * U < gs) load(k0 + 1024 * U);
        }
    } else {
        mx = max_xor(mx, 64);
        const float inv = (mx > 0.0f) ? 1.0f / mx : 0.0f;
        if (lane == 0) sg[u] = mx;
        for (int k = lane; k < gs; k += 64) dst[k] = qcode((float)src[k] * sr[k >> 6], inv);
    }
}

// Activations: fp32 rows -> per-(token, group) codes and scales; one block per (group, token) with the group's values
// in registers (quant_group). Bound by memory, 5 bytes per value: 4096 x 5120 35.6 us in two passes over the row,
// now 27. NV = 0: groups wider than 20480, in two passes.
template <int T, int NV>
__global__ __launch_bounds__(T) void k_quant_tok_grp(const float* x, int xstride, int K, int gs, int8_t* xq,
                                                     float* xs) {
    const int g = blockIdx.x, tok = blockIdx.y, t = threadIdx.x, ng = K / gs;
    __shared__ float red[T / 64];
    const float* row = x + (size_t)tok * xstride + (size_t)g * gs;
    int8_t* out = xq + (size_t)tok * K + (size_t)g * gs;
    if constexpr (NV > 0) {
        quant_group<T, NV>([&](int k) { return *(const float4*)(row + k); }, gs, 1.0f, out, xs + (size_t)tok * ng + g, red);
    } else {
        float mx = 0.0f;
        for (int k = 4 * t; k < gs; k += 4 * T) {
            const float4 v = *(const float4*)(row + k);
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
        mx = max_xor(mx, 64);
        if ((t & 63) == 0) red[t >> 6] = mx;
        __syncthreads();
        float m = red[0];
#pragma unroll
        for (int w = 1; w < T / 64; ++w) m = fmaxf(m, red[w]);
        const float sc = m * (1.0f / 127.0f), qi = (sc > 0.0f) ? 1.0f / sc : 0.0f;
        if (t == 0) xs[(size_t)tok * ng + g] = sc;
        for (int k = 4 * t; k < gs; k += 4 * T) {
            const float4 v = *(const float4*)(row + k);
            *(uint32_t*)(out + k) = pack4(qcode(v.x, qi), qcode(v.y, qi), qcode(v.z, qi), qcode(v.w, qi));
        }
    }
}
static int run_quant_tok_grp(const float* x, int xstride, int M, int K, int gs, int8_t* xq, float* xs, hipStream_t s) {
    const dim3 grid((unsigned)(K / gs), (unsigned)M);
#define Q27X_QT(T, NV) hipLaunchKernelGGL((k_quant_tok_grp<T, NV>), grid, dim3(T), 0, s, x, xstride, K, gs, xq, xs)
    if (gs <= 1024) Q27X_QT(256, 1);
    else if (gs <= 2048) Q27X_QT(256, 2);
    else if (gs <= 4096) Q27X_QT(256, 4);
    else if (gs <= 6144) Q27X_QT(512, 3);
    else if (gs <= 20480) Q27X_QT(1024, 5);
    else Q27X_QT(256, 0);
#undef Q27X_QT
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}

}  // namespace q27x

// ---------------------------------------------------------------- C ABI (prefill GEMM tier)
using namespace q27x;

extern "C" int q27x_i8g64_to_grp(const int8_t* w, const float* s64, int rows, int K, int gs, int8_t* wg,
                                 float* sg, q27x_stream_t s) {
    if (!w || !s64 || !wg || !sg || rows < 1 || K < 64 || gs < 64 || (gs & 63) || (K % gs)) {
        set_error("q27x_i8g64_to_grp: bad arguments (rows %d, K %d, gs %d)", rows, K, gs);
        return Q27X_E_ARG;
    }
    const dim3 grid((unsigned)(((long long)rows * (K / gs) + 3) / 4));
    if (!(((uintptr_t)w | (uintptr_t)wg) & 15))
        hipLaunchKernelGGL(k_i8g64_to_grp<true>, grid, dim3(256), 0, (hipStream_t)s, w, s64, rows, K, gs, wg, sg);
    else hipLaunchKernelGGL(k_i8g64_to_grp<false>, grid, dim3(256), 0, (hipStream_t)s, w, s64, rows, K, gs, wg, sg);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}

extern "C" int q27x_quant_tok_groups(const float* x, int xstride, int M, int K, int gs, int8_t* xq, float* xs,
                                     q27x_stream_t s) {
    if (!x || !xq || !xs || M < 1 || K < 4 || gs < 4 || (gs & 3) || (K % gs) || xstride < K || (xstride & 3) ||
        ((uintptr_t)x & 15)) {
        set_error("q27x_quant_tok_groups: bad arguments (M %d, K %d, gs %d, xstride %d)", M, K, gs, xstride);
        return Q27X_E_ARG;
    }
    return run_quant_tok_grp(x, xstride, M, K, gs, xq, xs, (hipStream_t)s);
}

extern "C" int q27x_gemm_i8g(const int8_t* w, const float* sw, int N, int K, int gs, float alpha, const int8_t* x,
                             const float* sx, int M, float* y, int ldy, const float* res, int ldr, float rs,
                             q27x_stream_t s) {
    if (!w || !sw || !x || !sx || !y || M < 1 || N < 1 || K < 1 || gs < 1 || ldy < N || (res && ldr < N)) {
        set_error("q27x_gemm_i8g: bad arguments");
        return Q27X_E_ARG;
    }
    if ((N % 128) || (K % kGK) || (gs % kGK) || (K % gs) || K / gs > kGMaxG || ((uintptr_t)w & 15) ||
        ((uintptr_t)x & 15)) {
        set_error("q27x_gemm_i8g: no kernel for N %d, K %d, gs %d (N %% 128, K %% %d, gs %% %d must be 0, "
                  "K/gs <= %d, 16-byte aligned codes)", N, K, gs, kGK, kGK, kGMaxG);
        return Q27X_E_SHAPE;
    }
    return launch_gemm_i8g(w, sw, N, K, gs, alpha, x, sx, M, y, ldy, 0, res, ldr, 0, rs, (hipStream_t)s);
}

namespace q27x {
static int g_gemm_cus = 0;
static int gemm_cus() {
    if (!g_gemm_cus) {
        int dev = 0;
        hipDeviceProp_t p;
        g_gemm_cus = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess &&
                      p.multiProcessorCount > 0) ? p.multiProcessorCount : 256;
    }
    return g_gemm_cus;
}
template <int WM, int WN, int KS, int S, bool GRP>
static int run_gemm_ring(const GemmArgs& a, hipStream_t s) {
    using C = RingCfg<WM, WN, KS, S>;
    const size_t lds = C::Ring + (size_t)(C::BM + C::BN) * a.ng * 4;
    if (lds > kSkLds) { set_error("gemm: no LDS for %d groups", a.ng); return Q27X_E_SHAPE; }
    static std::once_flag once;
    static hipError_t e = hipSuccess;
    std::call_once(once, [] {
        e = hipFuncSetAttribute((const void*)k_gemm_i8g_ring<WM, WN, KS, S, GRP>, hipFuncAttributeMaxDynamicSharedMemorySize, kSkLds);
    });
    Q27X_HIP(e);
    const unsigned grid = (unsigned)((a.N / C::BN) * ((a.M + C::BM - 1) / C::BM));
    hipLaunchKernelGGL((k_gemm_i8g_ring<WM, WN, KS, S, GRP>), dim3(grid), dim3(64 * C::NW), lds, s, a);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}
// the split-K kernel's launch: groups per phase by the LDS that their slots take beside the ring and the scales
template <int RT, int MT, int NW, int S>
static int run_gemm_sk(const GemmArgs& a, hipStream_t s) {
    using C = SkCfg<RT, MT, NW, S>;
    const size_t scl = (size_t)16 * (RT + MT) * a.ng * 4;
    const int cap = ((int)kSkLds - C::Ring - (int)scl) / (C::Out * 4);
    if (cap < 1) { set_error("gemm: no LDS for %d groups", a.ng); return Q27X_E_SHAPE; }
    const int ph = (a.ng + cap - 1) / cap, gpp = (a.ng + ph - 1) / ph;
    static std::once_flag once;
    static hipError_t e = hipSuccess;
    std::call_once(once, [] {
        e = hipFuncSetAttribute((const void*)k_gemm_i8g_sk<RT, MT, NW, S>, hipFuncAttributeMaxDynamicSharedMemorySize, kSkLds);
    });
    Q27X_HIP(e);
    const unsigned grid = (unsigned)((a.N / (16 * RT)) * ((a.M + 16 * MT - 1) / (16 * MT)));
    hipLaunchKernelGGL((k_gemm_i8g_sk<RT, MT, NW, S>), dim3(grid), dim3(64 * NW), C::Ring + scl + (size_t)gpp * C::Out * 4, s, a, gpp);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}
template <bool BF>
static int run_gemm_w4(const GemmArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((a.N / kW4B) * ((a.M + kW4B - 1) / kW4B)));
    if (!a.res) hipLaunchKernelGGL((k_gemm_i8g_w4<0, BF>), grid, dim3(512), 0, s, a);
    else if (!a.res_bf16) hipLaunchKernelGGL((k_gemm_i8g_w4<1, BF>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((k_gemm_i8g_w4<2, BF>), grid, dim3(512), 0, s, a);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}
template <bool BF>
static int run_gemm_rs(const GemmArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((a.N / kGN) * ((a.M + 255) / 256)));
    const size_t scl = (size_t)(256 + kGN) * a.ng * sizeof(float);
    if (!a.res) hipLaunchKernelGGL((k_gemm_i8g_rs<0, BF>), grid, dim3(512), scl, s, a);
    else if (!a.res_bf16) hipLaunchKernelGGL((k_gemm_i8g_rs<1, BF>), grid, dim3(512), scl, s, a);
    else hipLaunchKernelGGL((k_gemm_i8g_rs<2, BF>), grid, dim3(512), scl, s, a);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}

// The kernel forms and what a launch of each costs. A CU takes n = ceil(blocks / CUs) blocks, occ at a time; r blocks on
// a CU run their K / 128 (/ ks) stages and (with several groups) K / gs folds in T(r) = e + h r + stages t[r - 1] + folds
// g r us; all blocks together read (bm + bn) K bytes each at bw TB/s (100: no such bound seen), and the weights and
// outputs move at hb TB/s:
//   us = a + |(floor(n / occ) T(occ) + T(n % occ), blocks (bm + bn) K / bw, (N K + 4 M N) / hb)|
// (the root of the squares: the three overlap, but not fully where they are alike). The constants are fits of measured
// launches, on weights that a cache holds and on weights that none holds: 2941 shapes, M 1 to 4096, N 128 to 62080, K 128
// to 19200, one group and groups of 128 columns and more. The form taken is 0.5% (several groups) and 1.2% (one) off the
// fastest one on average. A cost without e, h and g, with constants from long K and groups of 1024 columns, was 5 to 6%
// off: it took split-K tiles of many short blocks, or too many folds, where larger tiles are up to 2.7 times as fast: us
// for 33 x 36864 x 512 27, now 10; 512 x 4096 x 256 in groups of 128 25 / 9; 384 x 14336 x 5120 in groups of 256 93 / 70.
// Against 128 x 128 tiles of 64-byte stages below 512 tokens and 256 x 128 or 256 x 256 ones from there: M = 1, 5120 x
// 17408: 86 / 20; M = 77: 102 / 33 (1024-column groups 125 / 45); M = 203, 34816 x 5120: 105 / 87; M = 512: 153 / 132;
// M = 1024, 5120 x 17408: 147 / 118.
enum { F_RING, F_SK, F_W4, F_RS, F_GEN };
struct GemmForm {
    int kind, bm, bn, ks, occ;
    float a, e, h, g, t[3], bw, hb;
    int (*run)(const GemmArgs&, hipStream_t);
};
static int run_w4(const GemmArgs& a, hipStream_t s) { return a.out_bf16 ? run_gemm_w4<true>(a, s) : run_gemm_w4<false>(a, s); }
static int run_rs(const GemmArgs& a, hipStream_t s) { return a.out_bf16 ? run_gemm_rs<true>(a, s) : run_gemm_rs<false>(a, s); }
// 64-byte stages: token tiles of 256 (8 waves, one block per CU, a 5-stage ring) or 128 (4 waves, two blocks per CU, a
// 4-stage ring, or 3 when 17+ groups' scales take the room)
static int run_gen256(const GemmArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)(a.N / kGN) * (unsigned)((a.M + 255) / 256));
    hipLaunchKernelGGL((k_gemm_i8g<256, 5>), grid, dim3(512), (size_t)(256 + kGN) * a.ng * sizeof(float), s, a);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}
static int run_gen128(const GemmArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)(a.N / kGN) * (unsigned)((a.M + 127) / 128));
    const size_t scl = (size_t)(128 + kGN) * a.ng * sizeof(float);
    if (64 * 1024 + scl <= 80 * 1024) hipLaunchKernelGGL((k_gemm_i8g<128, 4>), grid, dim3(256), scl, s, a);
    else hipLaunchKernelGGL((k_gemm_i8g<128, 3>), grid, dim3(256), scl, s, a);
    Q27X_HIP(hipGetLastError());
    return Q27X_OK;
}
// one group over K (the last three: shapes that the others do not take)
static const GemmForm kFormsK[] = {
    {F_SK, 16, 32, 4, 2, 2.10f, 1.50f, 0.09f, 0.00f, {0.355f, 0.641f}, 39.1f, 5.11f, run_gemm_sk<2, 1, 4, 3>},
    {F_SK, 32, 32, 4, 2, 1.69f, 1.49f, 0.67f, 0.00f, {0.420f, 0.793f}, 26.2f, 5.79f, run_gemm_sk<2, 2, 4, 2>},
    {F_SK, 32, 64, 4, 1, 1.25f, 4.26f, 0.00f, 0.00f, {0.694f}, 47.8f, 5.29f, run_gemm_sk<4, 2, 4, 2>},
    {F_RING, 64, 64, 1, 3, 2.10f, 1.38f, 0.95f, 0.00f, {0.300f, 0.460f, 0.605f}, 34.0f, 5.27f, run_gemm_ring<1, 1, 2, 3, false>},
    {F_RING, 64, 128, 1, 2, 1.83f, 0.80f, 2.16f, 0.00f, {0.298f, 0.566f}, 25.6f, 5.11f, run_gemm_ring<1, 2, 2, 3, false>},
    {F_RING, 64, 256, 1, 1, 0.11f, 5.32f, 0.00f, 0.00f, {0.623f}, 28.0f, 3.88f, run_gemm_ring<1, 4, 1, 3, false>},
    {F_RING, 128, 128, 1, 1, 0.00f, 4.58f, 0.00f, 0.00f, {0.399f}, 17.6f, 5.03f, run_gemm_ring<2, 2, 2, 3, false>},
    {F_RING, 128, 256, 1, 1, 0.11f, 5.74f, 0.00f, 0.00f, {0.805f}, 21.9f, 4.39f, run_gemm_ring<2, 4, 1, 3, false>},
    {F_RING, 256, 128, 1, 1, 0.19f, 6.21f, 0.00f, 0.00f, {0.689f}, 17.3f, 5.19f, run_gemm_ring<4, 2, 1, 3, false>},
    {F_W4, 256, 256, 1, 1, 0.25f, 7.61f, 0.00f, 0.00f, {1.300f}, 12.6f, 5.21f, run_w4},
    {F_GEN, 128, 128, 1, 2, 0.0f, 0.0f, 0.0f, 0.0f, {1.0f, 1.0f}, 100.0f, 5.0f, run_gen128},
    {F_GEN, 256, 128, 1, 1, 0.0f, 0.0f, 0.0f, 0.0f, {1.0f}, 100.0f, 5.0f, run_gen256},
    {F_RS, 256, 128, 1, 1, 0.0f, 0.0f, 0.0f, 0.0f, {1.0f}, 100.0f, 5.0f, run_rs},
};
// several groups
static const GemmForm kFormsG[] = {
    {F_SK, 16, 32, 4, 2, 0.95f, 1.89f, 0.41f, 0.24f, {0.352f, 0.829f}, 100.0f, 4.80f, run_gemm_sk<2, 1, 4, 3>},
    {F_SK, 32, 32, 8, 1, 1.10f, 2.01f, 0.00f, 0.27f, {0.830f}, 18.9f, 4.95f, run_gemm_sk<2, 2, 8, 2>},
    {F_SK, 32, 64, 4, 1, 1.32f, 3.24f, 0.00f, 0.69f, {0.715f}, 100.0f, 4.71f, run_gemm_sk<4, 2, 4, 2>},
    {F_RING, 64, 128, 1, 2, 2.91f, 1.73f, 0.09f, 1.17f, {0.438f, 0.934f}, 27.1f, 5.46f, run_gemm_ring<1, 2, 1, 3, true>},
    {F_RING, 64, 256, 1, 1, 0.59f, 3.83f, 0.00f, 1.38f, {0.565f}, 34.5f, 5.22f, run_gemm_ring<1, 4, 1, 3, true>},
    {F_RING, 128, 128, 1, 1, 0.32f, 4.61f, 0.00f, 1.22f, {0.476f}, 25.0f, 5.55f, run_gemm_ring<2, 2, 1, 4, true>},
    {F_RING, 128, 256, 1, 1, 0.06f, 4.98f, 0.00f, 0.92f, {0.729f}, 17.5f, 4.94f, run_gemm_ring<2, 4, 1, 3, true>},
    {F_RING, 256, 128, 1, 1, 0.15f, 4.97f, 0.00f, 0.98f, {0.668f}, 16.2f, 6.54f, run_gemm_ring<4, 2, 1, 3, true>},
    {F_RS, 256, 128, 1, 1, 2.08f, 3.24f, 0.00f, 1.05f, {0.810f}, 14.2f, 5.38f, run_rs},
    {F_GEN, 128, 128, 1, 2, 2.96f, 3.61f, 0.00f, 0.91f, {0.746f, 0.751f}, 14.4f, 5.10f, run_gen128},
    {F_GEN, 256, 128, 1, 1, 0.42f, 6.33f, 0.00f, 1.06f, {0.872f}, 14.0f, 4.85f, run_gen256},
};
// Whether the form takes the shape. The ring, split-K and 256 x 256 forms have whole 128-byte stages and 32-bit offsets
// of codes and outputs, k_gemm_i8g_rs 64-bit offsets of codes; k_gemm_i8g takes everything, and costs less than the
// others only with several small groups: with one group it is left the shapes that nothing else takes, token tiles of
// 256 from 512 tokens on.
static bool form_takes(const GemmForm& f, const GemmArgs& a) {
    if (a.N % f.bn) return false;
    const bool whole = a.K % 128 == 0 && a.gs % 128 == 0;
    const bool out32 = (long)a.M * a.ldy < (1L << 30) && (!a.res || (long)a.M * a.ldr < (1L << 30));
    const bool tiles = whole && out32 && (long)(a.M > a.N ? a.M : a.N) * a.K < (1L << 31);
    const bool rs = a.M >= 512 && a.K % 256 == 0 && whole && out32;
    switch (f.kind) {
        case F_W4: return tiles && a.M >= 512 && a.K >= 2 * kW4K;
        // three stages of 384 rows leave room for the scales of 10 groups
        case F_RING: return tiles && (f.bm + f.bn < 384 || a.ng <= 10);
        case F_SK: return tiles;
        case F_RS: return rs && (!tiles || a.ng > 1);
        default: return tiles ? a.ng > 1 : f.bm == 128 ? a.M < 512 : a.M >= 512 && !rs;
    }
}
static float form_cost(const GemmForm& f, const GemmArgs& a, int cus) {
    const long nb = (long)(a.N / f.bn) * ((a.M + f.bm - 1) / f.bm), n = (nb + cus - 1) / cus;
    const float stages = (float)(a.K / 128) / f.ks, folds = a.ng > 1 ? (float)a.ng : 0.0f, kb = (float)a.K * 1e-6f;
    auto T = [&](int r) { return f.e + f.h * r + stages * f.t[r - 1] + folds * f.g * r; };
    const int rem = (int)(n % f.occ);
    const float x = (float)(n / f.occ) * T(f.occ) + (rem ? T(rem) : 0.0f), y = (float)nb * (f.bm + f.bn) * kb / f.bw;
    const float z = (float)a.N * (kb + 4e-6f * a.M) / f.hb;
    return f.a + sqrtf(x * x + y * y + z * z);
}
// The form of a launch: the one that costs least. Q27X_GEMM_W4 = 1 / 0 takes / avoids the 256 x 256 tiles, Q27X_GEMM_FORM
// = i takes form i of the list, wherever the shape allows (tests of the kernels at small shapes, measurements).
static const GemmForm* pick_form(const GemmArgs& a, int* index) {
    const GemmForm* forms = a.ng == 1 ? kFormsK : kFormsG;
    const int nf = a.ng == 1 ? (int)(sizeof kFormsK / sizeof kFormsK[0]) : (int)(sizeof kFormsG / sizeof kFormsG[0]);
    const char* ew = getenv("Q27X_GEMM_W4");
    const char* ef = getenv("Q27X_GEMM_FORM");
    const bool force = ew && ew[0] == '1' && !ew[1], avoid = ew && ew[0] == '0' && !ew[1];
    const int want = ef && *ef ? atoi(ef) : -1;
    const GemmForm* best = nullptr;
    float cost = 0.0f;
    for (int i = 0; i < nf; ++i) {
        const GemmForm& f = forms[i];
        if (!form_takes(f, a) || (avoid && f.kind == F_W4)) continue;
        const float c = (i == want || (force && f.kind == F_W4)) ? -1.0f : form_cost(f, a, gemm_cus());
        if (!best || c < cost) { best = &f; cost = c; *index = i; }
    }
    return best;
}
static bool gemm_shape_ok(int M, int N, int K, int gs) {
    return M >= 1 && N >= 1 && K >= 1 && gs >= 1 && !(N % 128) && !(K % kGK) && !(gs % kGK) && !(K % gs) && K / gs <= kGMaxG;
}
int launch_gemm_i8g(const int8_t* w, const float* sw, int N, int K, int gs, float alpha, const int8_t* x,
                    const float* sx, int M, void* y, int ldy, int out_bf16, const void* res, int ldr, int res_bf16,
                    float rs, hipStream_t s, const AlphaSel* asel) {
    if (!gemm_shape_ok(M, N, K, gs) || ((uintptr_t)w & 15) || ((uintptr_t)x & 15) || ldy < N || (res && ldr < N)) {
        set_error("gemm: no kernel for M %d, N %d, K %d, gs %d", M, N, K, gs);
        return Q27X_E_SHAPE;
    }
    GemmArgs a{};
    a.w = w; a.sw = sw; a.x = x; a.sx = sx; a.y = (float*)y; a.res = (const float*)res; a.alpha = alpha; a.rs = rs;
    a.M = M; a.N = N; a.K = K; a.gs = gs; a.ng = K / gs; a.ldy = ldy; a.ldr = ldr;
    a.out_bf16 = out_bf16; a.res_bf16 = res_bf16;
    if (asel) a.asel = *asel;
    int form = 0;
    return pick_form(a, &form)->run(a, s);     // (a list's general forms take what its others do not)
}

}  // namespace q27x

extern "C" int q27x_gemm_i8g_form(int M, int N, int K, int gs, int* bm, int* bn) {
    if (!gemm_shape_ok(M, N, K, gs)) {
        set_error("q27x_gemm_i8g_form: no kernel for M %d, N %d, K %d, gs %d", M, N, K, gs);
        return Q27X_E_SHAPE;
    }
    GemmArgs a{};
    a.M = M; a.N = N; a.K = K; a.gs = gs; a.ng = K / gs; a.ldy = N;
    int form = 0;
    const GemmForm* f = pick_form(a, &form);
    if (bm) *bm = f->bm;
    if (bn) *bn = f->bn;
    return form;
}
