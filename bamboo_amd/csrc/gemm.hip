// MFMA GEMM for gfx950: bf16 (v_mfma_f32_16x16x32_bf16, v_mfma_f32_32x32x16_bf16) and fp32 (v_mfma_f32_16x16x4_f32, v_mfma_f32_32x32x2_f32, or six
// bf16 products of pieces), LDS-tiled, double-buffered, batched with two-level strides, fused epilogues.
//
// Stands in for F.linear / torch.matmul and their autograd backward in the reference layer
// (DeepSpeedExamples/pipeline_parallelism/transformer.py:121,127,136-146,158).
//
// bf16 data paths: NT and NN tiles by DMA on 16x16x32 instructions (gemm_m16.h), others on 32x32x16 (gemm_bf16_dma_*); 64x64 tiles with the
// contraction dealt to the waves (gemm_wave.h) for weight gradients of few tiles and few tiles of an odd contraction length; a register-staged
// kernel for rows of C that are no whole vectors (N % 8 != 0, NT).  fp32: gemm_f32.h, gemm_f32_pieces.hip.
#include "gemm_kernels.h"
#include "gemm_m16.h"
#include "gemm_f32.h"
#include "gemm_f32_pieces.h"
#include "gemm_wave.h"

// =========================================================================================
// host dispatch
// =========================================================================================
template <int BM, int BN, int WM, int WN>
static int launch_bf16(GemmArgs& g, int batches, hipStream_t st) {
    constexpr int smem = 2 * (BM + BN) * 64 * 2;
    auto kern = gemm_bf16_kernel<BM, BN, WM, WN>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    dim3 grid(g.tiles_m * g.tiles_n, 1, batches);
    bb_launch(kern, grid, dim3(WM * WN * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

template <int BM, int BN, int WM, int WN, bool AKM, bool BKM, bool DB, int STAGES = 4, int BK = 32, bool RAGK = false>
static int launch_bf16_dma(GemmArgs& g, int batches, hipStream_t st) {
    constexpr int smem = STAGES * (BM + BN) * BK * 2;
    auto kern = gemm_bf16_dma_kernel<BM, BN, WM, WN, AKM, BKM, DB, STAGES, BK, false, RAGK>;
    if constexpr (!AKM && !BKM) {       // dropout goes with forward (NT) products only: fill_args refuses the others
        if (g.drop.thresh) kern = gemm_bf16_dma_kernel<BM, BN, WM, WN, AKM, BKM, DB, STAGES, BK, true, RAGK>;
    }
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    dim3 grid(g.tiles_m * g.tiles_n, 1, batches);
    bb_launch(kern, grid, dim3(WM * WN * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// 256-row tiles: one block per CU walks the tiles; smaller ones, and a contraction of fewer k-tiles than the ring has stages: a block per tile.
static constexpr int kCUs = 256;
template <int TM, int TN, int WM, int WN, int STAGES, bool TB, bool WHOLE = false> static int launch_bf16_m16(GemmArgs& g, int batches, hipStream_t st) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16, smem = STAGES * (BM + BN) * 128;
    auto kern = gemm_bf16_m16_kernel<TM, TN, WM, WN, TB, STAGES, WHOLE, false>;
    if constexpr (!TB) {       // dropout goes with forward (NT) products only: fill_args refuses the others
        if (g.drop.thresh) kern = gemm_bf16_m16_kernel<TM, TN, WM, WN, TB, STAGES, WHOLE, true>;
    }
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int total = g.tiles_m * g.tiles_n, blocks = !WHOLE && BM == 256 && g.K >= STAGES * 64 && total > kCUs ? kCUs : total;
    bb_launch(kern, dim3(blocks, 1, batches), dim3(WM * WN * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

template <int BM, int BN, int WM, int WN, int STAGES = 3, bool WIDE = false>
static int launch_bf16_dma_stats(GemmArgs& g, hipStream_t st) {
    constexpr int smem = STAGES * (BM + BN) * 64 * 2;
    auto kern = gemm_bf16_dma_stats_kernel<BM, BN, WM, WN, STAGES, WIDE>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n), dim3(WM * WN * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

template <int BM, int BN, int WM, int WN, int STAGES = 3, bool WIDE = false>
static int launch_bf16_dma_bnbwd(GemmArgs& g, const BnBwdArgs& bn, hipStream_t st) {
    constexpr int smem = STAGES * (BM + BN) * 64 * 2;
    auto kern = gemm_bf16_dma_bnbwd_kernel<BM, BN, WM, WN, STAGES, WIDE>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n), dim3(WM * WN * 64), smem, st, g, bn);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// DMA kernels need at least one full vector of rows, and but for weight gradients and D128x128k64r K % 32 == 0; tile by problem size
enum DmaTile { D_NONE = 0, D256x256w8db, D256x128w8db, D128x128s3, D256x256k64, D256x128k64s3, D128x128k64, D128x64k64s3, D128x64s3,
               D64x128k64s3, D64x128s3, D256x192k64, D256x256p, D64x64k64s4, D128x128k64r, D128x128k64s3, D64x128k64s5, D256x128k64s2, D256x128k64w };
static const char* const kDmaTileNames[] = {"", "dma256x256w8db", "dma256x128w8db", "dma128x128s3", "dma256x256k64", "dma256x128k64s3",
                                            "dma128x128k64", "dma128x64k64s3", "dma128x64s3", "dma64x128k64s3", "dma64x128s3",
                                            "dma256x192k64", "dma256x256p", "dma64x64k64s4", "dma128x128k64r", "dma128x128k64s3", "dma64x128k64s5", "short_dma256x128k64s3",
                                            "whole_dma256x128k64s3"};
// The kernel of a bf16 problem depends on its shape, layout, output type and epilogue only (never on the stream, the environment or what
// ran before).  All tiles below add up a contraction in the same order, whichever runs changes no bit; the wave-sliced kernels (pick_wave)
// in another, and which of the two orders a problem has is its shape and layout alone: a redundant forward and a normal forward of the
// same layer give the same bits.  (fp32: shape and layout, the caller's word that pieces may be used, and their alignment, see pick_pieces.)
static DmaTile pick_dma_tile(int M, int N, int K, int64_t batches, int layout) {
    //  - Problems of at most one 64x64 tile per CU take those, four stages deep: what such a launch waits for is the chain of
    //    its k-tiles and its epilogue, and the more CUs share the loads the shorter both are.  128x64 / 64x64 tiles (us, back
    //    to back): NT 640x1024x4096 (160 tiles of 64x64) 24.1 / 16.4, 2048x1024x4096 (512) 26.3 / 27.9, 1500x1344x448 (504) 6.5 /
    //    7.5; NN 24.2 / 17.1, 25.5 / 29.8, 8.5 / 7.6.  One-wave tiles of 32x32 on four times the CUs: slower everywhere (100x1600x6400
    //    21.4 / 24.0), a wave has too many transfers to issue.  The shapes the larger tiles do not take (fewer than 128
    //    rows or columns) run on it too.
    const int64_t t64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64) * batches;
    if (layout != BB_TN && K % 64 == 0 && K > 0 && N % 8 == 0 && (t64 <= 256 || M < 128 || N < 128)) return D64x64k64s4;
    if ((K % 32 != 0 && layout != BB_TN) || K < 64 || M < 128 || N < 128 || N % 8 != 0) {
        //  - What is left goes to the wave-sliced 64x64 tiles (pick_wave) while these are at most two per CU, i.e. one round of
        //    them.  Beyond that they read more and hide less than 128x128 tiles with a masked last k-tile (us, 64x64 / 128x128):
        //    NT 2048x1000x1000 (512 tiles) 13.2 / 14.4, 4096x1000x1000 21.9 / 17.7, 8192x4096x72 67 / 30, 8192x4096x4008 499 / 316;
        //    NN 8192x1000x4008 132 / 78; 48 heads, NN 1032x80x1032 50 / 34, NT 1032x1032x80 111 / 55; TN 1032x80x1032 53 / 39.
        //    (An empty contraction has no k-tile to start with: the wave-sliced tiles go straight to their epilogue.)
        if (N % 8 != 0 || t64 <= 512 || K == 0) return D_NONE;
        if (layout != BB_TN) return D128x128k64r;
        return K >= 64 ? D128x128s3 : D_NONE;
    }
    // Rules read off sweeps of M 2048..16384 x N 768..6400 x K 1024/4096 (NT and NN) on MI355X (256 CUs,
    // one block of the 256-row tiles per CU).
    //  - Operands whose rows are k-contiguous (both of NT, A of NN) load faster as 64-wide k-tiles: one
    //    DMA instruction then covers 8 whole 128-byte lines instead of 16 half lines (128x128 tiles: up to +19 %).
    //  - 32-wide k-tiles (K % 64 != 0): above one round of 256x256 tiles they win while the last round is well filled; otherwise
    //    the small tiles, several blocks per CU, smooth the tail.  Within one round: 256x256 once 256x128 tiles would need a
    //    second round, 256x128 from about half a round on, and 128x128 tiles for anything smaller.
    const bool nt = layout == BB_NT, nn = layout == BB_NN;
    const bool k64 = (nt || nn) && K % 64 == 0 && K >= 128;
    const DmaTile small = k64 && (nt || K >= 2048) ? D128x128k64 : D128x128s3;
    const DmaTile mid = !k64 ? D256x128w8db : D256x128k64s3;
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((N + 255) / 256) * batches;
    const int64_t t2128 = (int64_t)((M + 255) / 256) * ((N + 127) / 128) * batches;
    const int64_t t128 = (int64_t)((M + 127) / 128) * ((N + 127) / 128) * batches;
    const bool big_ok = M >= 256 && N >= 256;
    //  - Problems of at most one half tile per CU take those: forward 128x64, from K 768 on 64x128, from 1536 on those of five stages, or 128x64
    //    where only these fit into a round; NN 64x128.  us, plain or with a residual (+):
    //        NT, both fit, 128x64 / 64x128           1050x1536x512 6.6* / 6.6    12168x128x512 5.3* / 5.3    6272x256x1024 8.4 / 7.1*    2043x768x768 6.5 / 6.2*
    //        NT, one fits, 128x64 / 128x128          627x3264x960+ 9.3* / 10.8   4427x448x1088+ 12.4* / 14.0   8680x192x7040+ 55.7* / 61.9
    //        NT, 64x128 of three stages / of five    2048x768x1024 7.1* / 7.3    1200x1600x1600+ 11.4 / 11.1*   2043x768x3072+ 17.6 / 16.6*   2048x1024x4096 22.7 / 22.1*
    //    Then 128x128 tiles of three stages, one per CU, up to a round of them.  The better half / 128x128:
    //        more than one half per CU, activation   1200x2048x512 9.6 / 9.1*    1600x2048x640 11.5 / 10.6*    3136x1024x256 8.5 / 8.0*    8112x512x128 8.2 / 7.9*
    //        NN, times a tensor                      1200x2048x512 8.1 / 7.7*    1600x2048x640 9.9 / 8.9*      3136x1024x256 6.6 / 6.5*    4096x768x3072 28.2 / 22.9*
    //        within a round of halves                2043x768x768 6.2* / 8.2     2048x1024x1024 7.3* / 9.6
    //        (a few rows, many columns, 256x128 / 128x128   640x6400x1600 24.1 / 17.3*)
    //    Larger ones: 256x128 and larger tiles, also for short contractions (NT 6272x1024x256 with activation 12.7, on 128x128 13.5), but halves for
    //    what has one to three k-tiles forward, where the launch is its epilogue (with activation, 128x64 / 128x128: 25088x512x128 19.5 / 22.2,
    //    6272x1024x128 11.9 / 12.3), or few columns.
    //    32-wide k-tiles (K % 64 != 0) as before: 128x64 tiles up to 128 tiles of 128x128 and for short forward contractions.
    if (k64) {
        const int64_t talls = (int64_t)((M + 127) / 128) * ((N + 63) / 64) * batches, flats = (int64_t)((M + 63) / 64) * ((N + 127) / 128) * batches;
        const bool tall = nt && (K < 768 || (flats > kCUs && talls <= kCUs));
        const int64_t halves = tall ? talls : flats;
        const DmaTile half = tall ? D128x64k64s3 : nt && K >= 1536 ? D64x128k64s5 : D64x128k64s3;
        if (halves <= kCUs) return half;
        if (t128 <= kCUs) return D128x128k64s3;
        if ((nt && K < 256) || (K < 768 && halves <= (K >= 512 ? 400 : 512))) return half;
    } else {
        if ((K <= 512 || t128 <= 128) && nt) return D128x64s3;
        if (t128 <= 128 && nn) return D64x128s3;
    }
    //  - Larger ones, whole 64-wide k-tiles: the tile of gemm_m16.h whose rounds take least, a round (one tile a CU) of kt k-tiles being
    //    kt times a step, plus what a tile costs around its loop (prologue, epilogue, the stores of all CUs at once).  Steps and rest as fitted
    //    to the table (a step of 256x256 is 1500 TFLOP/s).  Before (32x32x16 instructions, several kernels and rules) / 256x256 /
    //    256x192 / 256x128 (us, plain, the one taken marked):
    //        NT 8192x3072x1024 66 / 58 / 50* / 48    8192x4096x1024 78 / 63* / 66 / 66    8192x1024x4096 66 / 80 / 69 / 58*
    //           8192x1024x1024 24 / 29 / 25 / 22*    4096x4800x1600 73 / 73 / 60* / 62    4096x6400x1600, activation 97 / 85* / 101 / 97
    //           4096x1600x6400 86 / 117 / 97 / 76*
    //        NN 8192x4096x1024 77 / 62* / 67 / 67    8192x1024x4096 65 / 77 / 69 / 57*    8192x1024x3072 50 / 61 / 54 / 45*
    //           4096x1600x4800 67 / 87 / 76 / 59*    4096x6400x1600, times a tensor 95 / 81* / 99 / 97
    if (k64 && big_ok) {
        static const struct {
            DmaTile tile;
            int bn;
            double step, rest;
        } tiles[] = {{D256x256k64, 256, 1.36, 8.2}, {D256x192k64, 192, 1.05, 5.9}, {D256x128k64s3, 128, 0.755, 4.2}};
        DmaTile best = D_NONE;
        double least = 0.0;
        for (const auto& t : tiles) {
            const int64_t n = (int64_t)((M + 255) / 256) * ((N + t.bn - 1) / t.bn) * batches;
            const double us = (double)((n + 255) / 256) * (K / 64 * t.step + t.rest);
            if (best == D_NONE || us < least) best = t.tile, least = us;
        }
        return best;
    }
    if (t256 > 256) {
        const int64_t slots = (t256 + 255) / 256 * 256;
        const bool full70 = t256 * 10 >= slots * 7;
        if (!big_ok) return small;
        return full70 || K >= 1536 ? D256x256w8db : small;
    }
    if (big_ok && t2128 > 256) return D256x256w8db;
    if (M >= 256 && t2128 > 136) return mid;
    return small;
}

// ... of a problem with an fp32 output: of the tiles of gemm_m16.h, 256x128 has the registers for it.  ... and by what the epilogue reads (input
// gradients; us, before this rule / with it):
//  - Two operands, a few k-tiles, on 256x192 tiles: these wait for the second operand row by row; 128x128 tiles have other blocks to go on with.
//    15600x1088x192 43.2 / 35.6, 3999x4288x256 44.5 / 36.7, 4796x4608x384 51.8 / 49.3; K 448 0.96, 512 0.95 (9196x2048x512 54.6 / 49.8), 576 1.02.
//  - One operand to multiply by, up to twelve k-tiles, at most a round of 256x256 tiles: on the 32x32x16 loop, whose epilogue goes through LDS.  Multiplied
//    by a tensor, mean of 440 products, 16x16x32 / 32x32x16: K 128 1.037 / 1.012, 320..384 1.027 / 1.003, 576..768 1.019 / 1.009, 800..1100 1.011 / 1.009
//    (of the time before 16x16x32); masked by sign 0.99 / 1.01, plain 0.91 / 1.02, more than a round 0.96 / 0.95.
//  - Few k-tiles in a round of 256x128 tiles.  NN, two or three: two stages instead of three ("short_"), as the third's transfers would only be in the way of the
//    first's.  Up to eleven: fragments a whole k-tile ahead ("whole_"), but where GELU and its derivative want the registers.  Of the time on the 32x32x16 loop
//    before, half a k-tile ahead / two stages / whole (mean of 3000 products):
//        NN plain, K 128 1.015 / 0.983* / 1.024     192 1.024 / 0.987* / 1.022     256 1.019 / 1.005 / 1.010*      320..448 1.009 / 1.025 / 0.998*     512..704 0.995 / 1.065 / 0.981*
//        times a tensor  0.971 / 0.947* / 0.953     0.989 / 0.967* / 0.952         0.991 / 0.989 / 0.957*          0.981 / 1.018 / 0.945*              0.984 / 1.080 / 0.953*
//        NT residual                                                               0.979 / 0.984 / 0.949*          0.993 / 1.039 / 0.958*              0.974 / 1.074 / 0.949*
//        NT GELU and derivative                                                    0.922* / 0.922 / 0.984          0.934* / 0.971 / 0.983              0.941* / 1.028 / 0.988
//    (operands and outputs not in the last-level cache: 5054x1024x256 10.15 / 10.07 / 10.06 us, before 9.65; 13362x320x320 11.85 / 12.33 / 11.49, 11.25)
static DmaTile pick_dma_tile_for(int M, int N, int K, int64_t batches, int layout, bool c_f32, int epilogue, bool resid) {
    const DmaTile t = pick_dma_tile(M, N, K, batches, layout);
    if (c_f32 && (t == D256x256k64 || t == D256x192k64)) return D256x128k64s3;
    if (t == D256x192k64 && layout == BB_NN && K <= 512 && epilogue == BB_EPI_MUL_POS && resid) return D128x128s3;
    if (t == D256x256k64 && layout == BB_NN && K <= 768 && epilogue == BB_EPI_MUL && (int64_t)((M + 255) / 256) * ((N + 255) / 256) * batches <= kCUs) return D256x256w8db;
    if (t == D256x128k64s3 && K < 768 && (int64_t)((M + 255) / 256) * ((N + 127) / 128) * batches <= kCUs) {
        if (layout == BB_NN && K <= 192) return D256x128k64s2;
        if (epilogue != BB_EPI_ACT_DACT) return D256x128k64w;
    }
    // (more than one 256x256 tile of a batch a CU goes by a name of its own: the blocks then walk their batch's tiles; so do those of the other two)
    return t == D256x256k64 && (int64_t)((M + 255) / 256) * ((N + 255) / 256) > kCUs ? D256x256p : t;
}

// The kernels that leave column statistics (128x64, 64x128 or 256x128 tiles) take the largest within a round of them and, forward, where its
// rounds are filled and those of 256x256 tiles are not.
static bool stats_256x128(DmaTile t, int M, int N, int layout) {
    if (t != D256x256k64 && t != D256x192k64 && t != D256x128k64s3) return false;
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((N + 255) / 256), t2128 = (int64_t)((M + 255) / 256) * ((N + 127) / 128);
    if (t2128 <= 256) return t2128 > 136;
    const int64_t slots = (t256 + 255) / 256 * 256, slots2 = (t2128 + 255) / 256 * 256;
    return layout == BB_NT && t256 > 256 && t256 * 100 < slots * 85 && t2128 * 10 >= slots2 * 9;
}

// NT and NN kernels reach a tile's rows by 32-bit offsets (DmaLanes); operands whose rows lie further apart take the kernel with
// an address per lane.
static DmaTile narrow_or_wide(DmaTile t, int layout, int64_t lda, int64_t ldb) {
    return t != D_NONE && layout != BB_TN && (lda >= kDmaMaxLd || ldb >= kDmaMaxLd) ? D128x128k64r : t;
}

// The wave-sliced kernels (gemm_wave.h) take the weight gradients whose 64x64 tiles are at most one per CU, and what the
// DMA kernels do not take (contractions of odd lengths, few tiles).  W_8: eight waves, 32-wide slices, two stages each (130 KB of LDS);
// W_4: four waves, 64-wide slices, one stage (65 KB, two blocks a CU).  Measured back to back, 128x128 DMA tiles / W_8 (us):
// TN 512x512x4096 55.7 / 18.8, 256x256x6272 80.8 / 21.9; register-staged kernel / W_8: NT 200x264x72 31.4 / 5.2.
enum WaveMode { W_NONE = 0, W_8, W_4 };
static WaveMode pick_wave(int M, int N, int K, int64_t batches, int layout, DmaTile dma) {
    if (N % 8 != 0) return W_NONE;
    const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64) * batches;
    if (dma != D_NONE && (tiles > 256 || layout != BB_TN)) return W_NONE;
    return tiles <= 256 ? W_8 : W_4;
}
template <bool TA, bool TB, int KW, int BK, int NST> static int launch_bf16_wave(GemmArgs& g, int batches, hipStream_t st) {
    auto kern = gemm_bf16_wave_kernel<TA, TB, KW, BK, NST, false>;
    if constexpr (!TA && !TB) {
        if (g.drop.thresh) kern = gemm_bf16_wave_kernel<TA, TB, KW, BK, NST, true>;
    }
    constexpr int smem = wave_gemm_lds(KW, BK, NST);
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + 63) / 64;
    g.tiles_n = (g.N + 63) / 64;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n, 1, batches), dim3(KW * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// 64x64 tiles that are at most half of the CUs' go as two blocks a tile, 32x64 and four waves each, of 16x32 (gemm_m16.h; the same bits): a CU has half
// the LDS reads and transfers to get through in a k-tile.  Before (two waves, 32x32x16 instructions) / now, us: NN 128x256x128 3.3 / 3.0, 1024x512x512 (128
// tiles) 4.4 / 3.8, x2048 8.8 / 6.9, 512x768x3072 11.6 / 9.0, 300x1600x1600 7.4 / 6.0; NT 3.7 / 3.3, 4.3 / 3.8, 8.6 / 6.8, 11.3 / 8.6, 7.3 / 5.9.  More
// halves than CUs, 64x64 / halves: NN 1050x512x2048 (136 tiles) 9.1 / 9.3, NT 8.3 / 9.0, 2048x512x512 (256) 4.5 / 4.8.  NT 64x64 tiles have eight
// waves of 16x32 (four on 32x32x16 / this: 1050x512x512 4.5 / 4.3, x2048 8.5 / 8.3, 1024x1024x512 with activation 5.7 / 5.2, 640x1024x4096
// 14.8 / 14.8), NN ones four of 32x32 (9.1 / 9.9, 15.9 / 17.0: the four waves of a column each read its k-major fragments, two reads apiece).
static bool halve_tiles(int M, int N, int64_t batches) { return (int64_t)((M + 31) / 32) * ((N + 63) / 64) * batches <= 256; }

template <bool TA, bool TB> static int dispatch_bf16(GemmArgs& g, int batches, hipStream_t st) {
    const int layout = TA ? BB_TN : TB ? BB_NN : BB_NT;
    const DmaTile dma = narrow_or_wide(pick_dma_tile_for(g.M, g.N, g.K, batches, layout, g.c_f32 != 0, g.epilogue, g.resid != nullptr), layout, g.lda, g.ldb);
    switch (pick_wave(g.M, g.N, g.K, batches, layout, dma)) {
        case W_8: return launch_bf16_wave<TA, TB, 8, 32, 2>(g, batches, st);
        case W_4: return launch_bf16_wave<TA, TB, 4, 64, 1>(g, batches, st);
        default: break;
    }
    switch (dma) {
        case D256x256w8db: return launch_bf16_dma<256, 256, 2, 4, TA, TB, true>(g, batches, st);
        case D256x128w8db: return launch_bf16_dma<256, 128, 4, 2, TA, TB, true>(g, batches, st);
        case D128x128s3: return launch_bf16_dma<128, 128, 2, 2, TA, TB, true, 3>(g, batches, st);
        case D256x256k64:
        case D256x256p:
            if constexpr (!TA) return launch_bf16_m16<8, 4, 2, 4, 2, TB>(g, batches, st);
            else break;
        case D256x192k64:
            if constexpr (!TA) return launch_bf16_m16<4, 6, 4, 2, 2, TB>(g, batches, st);
            else break;
        case D256x128k64s3:
            if constexpr (!TA) return launch_bf16_m16<4, 4, 4, 2, 3, TB>(g, batches, st);
            else break;
        case D256x128k64w:
            if constexpr (!TA) return launch_bf16_m16<4, 4, 4, 2, 3, TB, true>(g, batches, st);
            else break;
        case D256x128k64s2:
            if constexpr (TB && !TA) return launch_bf16_m16<4, 4, 4, 2, 2, TB>(g, batches, st);
            else break;
        case D128x128k64: return launch_bf16_dma<128, 128, 2, 2, TA, TB, true, 2, 64>(g, batches, st);
        case D128x128k64r:
            if constexpr (!TA) return launch_bf16_dma<128, 128, 2, 2, TA, TB, true, 2, 64, true>(g, batches, st);
            else break;
        case D128x128k64s3:
            if constexpr (!TA) return launch_bf16_m16<4, 2, 2, 4, 3, TB, true>(g, batches, st);
            else break;
        case D128x64k64s3:
            if constexpr (!TA && !TB) return launch_bf16_m16<2, 2, 4, 2, 3, TB, true>(g, batches, st);
            else break;
        case D128x64s3: return launch_bf16_dma<128, 64, 4, 1, TA, TB, true, 3>(g, batches, st);
        case D64x128k64s3:
            if constexpr (!TA) return launch_bf16_m16<2, 2, 2, 4, 3, TB>(g, batches, st);
            else break;
        case D64x128k64s5:
            if constexpr (!TA && !TB) return launch_bf16_m16<2, 2, 2, 4, 5, TB, true>(g, batches, st);
            else break;
        case D64x128s3: return launch_bf16_dma<64, 128, 2, 2, TA, TB, true, 3>(g, batches, st);
        case D64x64k64s4:
            if constexpr (!TA)
                return halve_tiles(g.M, g.N, batches) ? launch_bf16_m16<1, 2, 2, 2, 4, TB, true>(g, batches, st)
                       : TB ? launch_bf16_dma<64, 64, 2, 2, TA, true, true, 4, 64>(g, batches, st) : launch_bf16_m16<1, 2, 4, 2, 4, false, true>(g, batches, st);
            else break;
        default: break;
    }
    if constexpr (!TA && !TB) return launch_bf16<128, 128, 2, 2>(g, batches, st);
    bb_set_error("bb_gemm: no kernel for this problem");   // N % 8 == 0 is checked for the other layouts
    return BB_EINVAL;
}

// fp32 problems of few tiles and a contraction of at most one slice a wave (the products of attention heads, the input gradients
// of a narrow model, weight gradients over few rows) take 32x32 tiles, up to four per CU.  64x64 tiles / this (us, back to
// back): NN 128x128x128 6.6 / 3.9, 512x1024x64 5.4 / 4.6, 2048x384x128 (768 tiles) 7.2 / 6.1, 2048x512x128 (1024) 7.3 / 7.0,
// 2048x1024x128 (2048) 9.9 / 11.6.  Weight gradients share a launch with the others of their layer, so there the limit is
// each problem's own (a problem gives the same bits alone and in a group): 128 rows x 128 (x 2 in the feed-forward) 7.8 / 4.8,
// x 256 (x 4) 8.4 / 6.8, x 384 (576 tiles the largest) 11.0 / 12.2.  The layers' own forward products (NT, unbatched), whose last
// bits decide ReLUs, keep the order of additions of the larger tiles, as in bf16.
static bool pick_f32_wave(int M, int N, int K, int64_t batches, int layout) {
    const int64_t tiles = (int64_t)((M + 31) / 32) * ((N + 31) / 32) * batches;
    if (layout == BB_NT && batches == 1) return false;
    return K <= kF32WaveK && tiles <= (layout == BB_TN && batches == 1 ? 256 : 1024);
}
// problems of longer contractions on shared ones, see pick_f32_split
static constexpr int kF32SplitGroups = 2, kF32SplitBN = 32;
// Of what is left for the tiles of 64x64 and 64x32, problems of at most 128 64x64 tiles take four blocks a tile instead, with the
// same bits (gemm_f32_quarter_kernel): until then every CU has at most two of them.  Larger tiles / this (us, back to back): NT
// 128x128x128 7.0 / 5.2, 512x512x256 (64 tiles) 10.7 / 5.8, 1000x448x448 (112) 16.3 / 10.2, 1024x512x512 (128) 11.2 / 11.4,
// 1024x512x2048 32.3 / 29.9, 512x1536x256 (192) 11.4 / 11.2, 1000x1344x448 (336) 25.1 / 26.8, 2048x768x768 (384) 29.0 / 37.9; NN
// alike.  TN: 64x64x4096 85 / 41, 512x512x2048 45 / 24, 512x1024x1000 (128) 25.2 / 18.3; the weight gradients of a layer
// together, hidden size (x 4 in the feed-forward) and rows: 128 (48 tiles) 7680 159 / 80, 200 10.7 / 7.5; 192 (108) 3000 67 / 46;
// 256 (192) 1072 29.4 / 31.2, 320 (300) 600 28.2 / 31.6; ResNet blocks of 64 channels (17) 6272 pixels 131 / 65.
static constexpr int kF32QuarterTiles = 128;
static bool pick_f32_quarter(int M, int N, int64_t batches) { return (int64_t)((M + 63) / 64) * ((N + 63) / 64) * batches <= kF32QuarterTiles; }
template <bool TA, bool TB, int KG> static int launch_f32_quarter(GemmArgs& g, int batches, hipStream_t st) {
    auto kern = gemm_f32_quarter_kernel<TA, TB, KG>;
    g.tiles_m = (g.M + 31) / 32;
    g.tiles_n = (g.N + 31) / 32;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n, 1, batches), dim3(256 * KG), kF32QuarterLds, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
template <bool TA, bool TB> static int launch_f32_wave(GemmArgs& g, int batches, hipStream_t st) {
    auto kern = gemm_f32_wave_kernel<TA, TB>;
    g.tiles_m = (g.M + 31) / 32;
    g.tiles_n = (g.N + 31) / 32;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n, 1, batches), dim3(kF32Waves * 64), kF32WaveLds, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
// rows too wide for the kernels' 32-bit offsets inside a tile (64 rows of 2^22 elements are 2^30 bytes): 64x64 tiles with 64-bit ones
static bool f32_wide(int64_t lda, int64_t ldb) { return lda >= (1 << 22) || ldb >= (1 << 22); }
template <bool TA, bool TB, int BN, bool WIDE = false> static int launch_f32(GemmArgs& g, int batches, hipStream_t st) {
    g.tiles_m = (g.M + 63) / 64;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch((gemm_f32_kernel<TA, TB, BN, WIDE>), dim3(g.tiles_m * g.tiles_n, 1, batches), dim3(256), f32_gemm_lds(BN), st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
template <bool TA, bool TB> static int dispatch_f32(GemmArgs& g, int batches, hipStream_t st) {
    if (f32_wide(g.lda, g.ldb)) return launch_f32<TA, TB, 64, true>(g, batches, st);
    if (pick_f32_wave(g.M, g.N, g.K, batches, TA ? BB_TN : TB ? BB_NN : BB_NT)) return launch_f32_wave<TA, TB>(g, batches, st);
    const bool split = pick_f32_split(g.M, g.N, g.K, batches, TA ? BB_TN : TB ? BB_NN : BB_NT);
    const bool quarter = pick_f32_quarter(g.M, g.N, batches);
    if (quarter && !split) return launch_f32_quarter<TA, TB, 1>(g, batches, st);
    if constexpr (!TA) {
        if (split) return quarter ? launch_f32_quarter<TA, TB, 2>(g, batches, st) : launch_f32<TA, TB, kF32SplitBN>(g, batches, st);
    }
    return launch_f32<TA, TB, 64>(g, batches, st);
}

extern "C" int bb_gemm_variant(const bb_gemm_desc* d, char* out, int out_len) {
    BB_REQUIRE(d && out && out_len > 0, "bb_gemm_variant: bad arguments");
    static const char* const layouts[] = {"nt", "nn", "tn"};
    BB_REQUIRE(d->layout >= BB_NT && d->layout <= BB_TN, "bb_gemm_variant: bad layout %d", d->layout);
    const int64_t batches = (int64_t)(d->nb1 > 0 ? d->nb1 : 1) * (d->nb2 > 0 ? d->nb2 : 1);
    if (d->dtype == BB_BF16) {
        const DmaTile dt = narrow_or_wide(pick_dma_tile_for(d->M, d->N, d->K, batches, d->layout, d->c_dtype == BB_F32, d->epilogue, d->resid != nullptr), d->layout, d->lda, d->ldb);
        const WaveMode wm = pick_wave(d->M, d->N, d->K, batches, d->layout, dt);
        if (wm != W_NONE) snprintf(out, out_len, "bf16_%s_wave64x64k%d", layouts[d->layout], wm == W_8 ? 8 : 4);
        else snprintf(out, out_len, "bf16_%s_%s%s", layouts[d->layout], dt == D64x64k64s4 && halve_tiles(d->M, d->N, batches) ? "halves_" : "",
                 dt != D_NONE ? kDmaTileNames[dt] : "128x128");
    }
    else if (const PiecesTile tile = pick_pieces(d, 1)) snprintf(out, out_len, "f32_%s_pieces128x%d", layouts[d->layout], tile == P128x128 ? 128 : 64);
    else if (f32_wide(d->lda, d->ldb)) snprintf(out, out_len, "f32_%s_64x64wide", layouts[d->layout]);
    else if (pick_f32_wave(d->M, d->N, d->K, batches, d->layout)) snprintf(out, out_len, "f32_%s_wave32x32k%d", layouts[d->layout], kF32Waves);
    else {
        const char* quarter = pick_f32_quarter(d->M, d->N, batches) ? "quarter" : "";
        if (pick_f32_split(d->M, d->N, d->K, batches, d->layout))
            snprintf(out, out_len, "f32_%s_%s64x%dk%d", layouts[d->layout], quarter, kF32SplitBN, kF32SplitGroups);
        else snprintf(out, out_len, "f32_%s_%s64x64", layouts[d->layout], quarter);
    }
    return BB_OK;
}

static int fill_args(const bb_gemm_desc* d, GemmArgs& g, int64_t& batches, bool& ta, bool& tb) {
    BB_REQUIRE(d != nullptr, "bb_gemm: null descriptor");
    BB_REQUIRE(d->dtype == BB_F32 || d->dtype == BB_BF16, "bb_gemm: bad dtype %d", d->dtype);
    BB_REQUIRE(d->c_dtype == d->dtype || d->c_dtype == BB_F32, "bb_gemm: bad c_dtype %d", d->c_dtype);
    BB_REQUIRE(d->layout >= BB_NT && d->layout <= BB_TN, "bb_gemm: bad layout %d", d->layout);
    BB_REQUIRE(d->M >= 0 && d->N >= 0 && d->K >= 0, "bb_gemm: negative dimension");
    BB_REQUIRE(!d->accumulate || d->c_dtype == BB_F32, "bb_gemm: accumulate needs an fp32 C");
    BB_REQUIRE(d->epilogue >= BB_EPI_NONE && d->epilogue <= BB_EPI_MUL_POS, "bb_gemm: bad epilogue");
    const int nb1 = d->nb1 > 0 ? d->nb1 : 1, nb2 = d->nb2 > 0 ? d->nb2 : 1;
    batches = (int64_t)nb1 * nb2;
    ta = d->layout == BB_TN;
    tb = d->layout != BB_NT;
    g.M = d->M; g.N = d->N; g.K = d->K; g.nb2 = nb2;
    if (d->M == 0 || d->N == 0) return BB_OK;
    BB_REQUIRE(d->A && d->B && d->C, "bb_gemm: null operand");
    BB_REQUIRE((d->epilogue != BB_EPI_DACT && d->epilogue != BB_EPI_MUL && d->epilogue != BB_EPI_MUL_POS && d->epilogue != BB_EPI_MUL_POS) || d->aux_in,
               "bb_gemm: DACT / MUL / MUL_POS epilogue needs aux_in");
    BB_REQUIRE(d->epilogue != BB_EPI_RESIDUAL || d->resid, "bb_gemm: RESIDUAL epilogue needs resid");
    BB_REQUIRE(d->epilogue != BB_EPI_ACT_DACT || d->aux_out, "bb_gemm: ACT_DACT epilogue needs aux_out");
    BB_REQUIRE(batches <= 65535, "bb_gemm: too many batches (%lld)", (long long)batches);
    const int vec = d->dtype == BB_BF16 ? 8 : 4;
    const bool conv = d->conv_c != 0 || d->conv_h != 0 || d->conv_w != 0 || d->conv_row0 != 0;
    if (conv) {
        // B = patch matrix of an NHWC tensor, gathered by the grouped DMA kernel's loader
        BB_REQUIRE(d->layout == BB_TN && d->dtype == BB_BF16 && batches == 1, "bb_gemm: a patch-matrix B needs BB_TN, bf16, no batching");
        BB_REQUIRE(d->conv_c > 0 && d->conv_c % 64 == 0 && d->conv_h > 0 && d->conv_w > 0 && d->conv_row0 >= 0,
                   "bb_gemm: patch-matrix B: conv_c (%d) must be a positive multiple of 64 (128x128 tiles take a multiple of 128), conv_h/conv_w positive", d->conv_c);
        BB_REQUIRE(d->N == 9 * d->conv_c, "bb_gemm: patch-matrix B: N (%d) must be 9 * conv_c (%d)", d->N, d->conv_c);
        BB_REQUIRE(32 / d->conv_w + 1 <= d->conv_h,
                   "bb_gemm: patch-matrix B: 32 pixels must not span more than one image boundary (%d x %d)", d->conv_h, d->conv_w);
        BB_REQUIRE(!d->bias && d->epilogue == BB_EPI_NONE, "bb_gemm: patch-matrix B takes no bias / epilogue");
    }
    // the contiguous dimension of every operand is read in 16-byte vectors
    const int a_contig = ta ? d->M : d->K, b_contig = conv ? d->conv_c : tb ? d->N : d->K;
    const int64_t ldb = conv ? d->conv_c : d->ldb;
    BB_REQUIRE(a_contig % vec == 0 && d->lda % vec == 0, "bb_gemm: A contiguous dim/lda must be a multiple of %d", vec);
    BB_REQUIRE(b_contig % vec == 0 && ldb % vec == 0, "bb_gemm: B contiguous dim/ldb must be a multiple of %d", vec);
    BB_REQUIRE(((uintptr_t)d->A % 16) == 0 && ((uintptr_t)d->B % 16) == 0, "bb_gemm: operands must be 16-byte aligned");
    BB_REQUIRE(d->sA1 % vec == 0 && d->sA2 % vec == 0 && d->sB1 % vec == 0 && d->sB2 % vec == 0,
               "bb_gemm: batch strides of A/B must be multiples of %d", vec);
    BB_REQUIRE(d->lda >= a_contig && ldb >= b_contig && d->ldc >= d->N, "bb_gemm: leading dimension too small");
    g.A = d->A; g.B = d->B; g.C = d->C;
    g.bias = d->bias; g.aux_in = d->aux_in; g.aux_out = d->aux_out; g.resid = d->resid;
    g.colsum = nullptr;
    BB_REQUIRE(!d->colsum_out || d->layout == BB_TN, "bb_gemm: colsum_out needs the BB_TN layout");
    g.lda = d->lda; g.ldb = ldb; g.ldc = d->ldc; g.ldaux = d->ldaux > 0 ? d->ldaux : d->ldc;
    g.conv_h = d->conv_h; g.conv_w = d->conv_w; g.conv_c = d->conv_c; g.conv_row0 = d->conv_row0;
    g.strip_stats = nullptr;   // bb_gemm sets it where the kernel that runs the problem produces them
    g.sA1 = d->sA1; g.sA2 = d->sA2; g.sB1 = d->sB1; g.sB2 = d->sB2; g.sC1 = d->sC1; g.sC2 = d->sC2;
    g.alpha = d->alpha;
    g.epilogue = d->epilogue; g.act = d->act; g.accumulate = d->accumulate;
    g.c_f32 = (d->c_dtype == BB_F32);
    BB_REQUIRE(d->dropout_p >= 0.f && d->dropout_p < 1.f, "bb_gemm: dropout_p must be in [0, 1)");
    BB_REQUIRE(d->dropout_p == 0.f || (batches == 1 && d->layout == BB_NT && d->epilogue != BB_EPI_DACT && d->epilogue != BB_EPI_MUL && d->epilogue != BB_EPI_MUL_POS &&
                                       !d->accumulate),
               "bb_gemm: dropout goes with an unbatched, non-accumulating NT problem and not with the DACT / MUL / MUL_POS epilogues");
    g.drop = bb_drop_key(d->dropout_p, d->dropout_k0, d->dropout_k1, (uint64_t)d->M * (uint64_t)d->N);
    g.tiles_m = g.tiles_n = 0;
    return BB_OK;
}

// The bias-gradient column sums ride inside the DMA and the wave-sliced kernels when they run the problem; otherwise
// the stand-alone reduction computes them.
static bool colsum_fusable(const bb_gemm_desc* d, int64_t batches) {
    if (!d->colsum_out || d->dtype != BB_BF16 || batches != 1) return false;
    const DmaTile dma = pick_dma_tile(d->M, d->N, d->K, 1, d->layout);
    return dma != D_NONE || pick_wave(d->M, d->N, d->K, 1, d->layout, dma) != W_NONE;
}
static int colsum_standalone(const bb_gemm_desc* d, void* stream) {
    BB_REQUIRE(d->colsum_ws, "bb_gemm: colsum_out on this problem needs colsum_ws");
    return bb_colsum_acc(d->dtype, d->K, d->M, d->A, d->lda, d->colsum_out, d->colsum_ws, stream);
}

extern "C" int bb_gemm_strip_stats_supported(const bb_gemm_desc* d) {
    return d && d->dtype == BB_BF16 && d->c_dtype == BB_BF16 && d->layout == BB_NT && d->nb1 <= 1 && d->nb2 <= 1 &&
           d->M >= 128 && d->N >= 64 && d->N % 8 == 0 && d->K >= 128 && d->K % 64 == 0 && d->conv_c == 0 && !d->colsum_out &&
           !d->bias && d->epilogue == BB_EPI_NONE && d->alpha == 1.0f && d->dropout_p == 0.f;
}
extern "C" int64_t bb_strip_stats_workspace(int rows, int cols) { return (int64_t)((rows + 31) / 32) * 3 * cols; }

extern "C" int64_t bb_bn_bwd_strips_workspace(int rows, int cols) { return (int64_t)((rows + 31) / 32) * 2 * cols; }

static int check_bn_bwd_stats(const char* name, const bb_bn_bwd_stats* bn) {
    BB_REQUIRE(bn && bn->x && bn->mean && bn->rstd && bn->strips, "%s: null pointer in bb_bn_bwd_stats", name);
    BB_REQUIRE(((uintptr_t)bn->x % 16) == 0 && ((uintptr_t)bn->mean % 16) == 0 && ((uintptr_t)bn->rstd % 16) == 0 &&
               ((uintptr_t)bn->strips % 16) == 0, "%s: the bb_bn_bwd_stats operands must be 16-byte aligned", name);
    return BB_OK;
}

extern "C" int bb_gemm_bn_bwd_supported(const bb_gemm_desc* d) {
    return d && d->dtype == BB_BF16 && d->c_dtype == BB_BF16 && d->layout == BB_NN && d->nb1 <= 1 && d->nb2 <= 1 &&
           d->M >= 128 && d->N >= 128 && d->N % 8 == 0 && d->K >= 128 && d->K % 64 == 0 && d->conv_c == 0 && !d->colsum_out &&
           !d->strip_stats && !d->bias && !d->accumulate && d->alpha == 1.0f && d->dropout_p == 0.f && d->ldc == d->N &&
           (d->ldaux == 0 || d->ldaux == d->N) &&
           (d->epilogue == BB_EPI_NONE || (d->epilogue == BB_EPI_RESIDUAL && d->resid) || (d->epilogue == BB_EPI_MUL_POS && d->aux_in));
}

extern "C" int bb_gemm_bn_bwd(const bb_gemm_desc* d, const bb_bn_bwd_stats* bn, void* stream) {
    BB_REQUIRE(bb_gemm_bn_bwd_supported(d), "bb_gemm_bn_bwd: needs an unbatched bf16 BB_NN problem with a contiguous bf16 C, M >= 128, "
               "N >= 128, N %% 8 == 0, K >= 128, K %% 64 == 0, alpha = 1, no bias, epilogue BB_EPI_NONE, BB_EPI_RESIDUAL or BB_EPI_MUL_POS");
    int rc = check_bn_bwd_stats("bb_gemm_bn_bwd", bn);
    if (rc) return rc;
    GemmArgs g;
    int64_t batches;
    bool ta, tb;
    rc = fill_args(d, g, batches, ta, tb);
    if (rc) return rc;
    const BnBwdArgs b = {bn->x, bn->mean, bn->rstd, bn->strips};
    const DmaTile dma = narrow_or_wide(pick_dma_tile(d->M, d->N, d->K, 1, BB_NN), BB_NN, g.lda, g.ldb);
    if (dma == D128x128k64r) return launch_bf16_dma_bnbwd<64, 128, 2, 2, 3, true>(g, b, (hipStream_t)stream);
    if (dma == D64x64k64s4) return launch_bf16_dma_bnbwd<64, 64, 2, 2, 4>(g, b, (hipStream_t)stream);
    if (stats_256x128(dma, g.M, g.N, BB_NN)) return launch_bf16_dma_bnbwd<256, 128, 4, 2>(g, b, (hipStream_t)stream);
    return launch_bf16_dma_bnbwd<64, 128, 2, 2>(g, b, (hipStream_t)stream);
}

extern "C" int bb_gemm(const bb_gemm_desc* d, void* stream) {
    if (d && d->conv_c != 0) return bb_gemm_grouped(d, 1, stream);   // only the grouped kernel gathers a patch-matrix B
    if (d && d->strip_stats) {
        BB_REQUIRE(bb_gemm_strip_stats_supported(d), "bb_gemm: strip_stats needs an unbatched bf16 BB_NT problem with a bf16 C, "
                   "M >= 128, N >= 64, N %% 8 == 0, K >= 128, K %% 64 == 0, alpha = 1, no bias, no epilogue");
        BB_REQUIRE(((uintptr_t)d->strip_stats % 16) == 0, "bb_gemm: strip_stats must be 16-byte aligned");
        GemmArgs g;
        int64_t batches;
        bool ta, tb;
        int rc = fill_args(d, g, batches, ta, tb);
        if (rc) return rc;
        g.strip_stats = d->strip_stats;
        const DmaTile dma = narrow_or_wide(pick_dma_tile(d->M, d->N, d->K, 1, BB_NT), BB_NT, g.lda, g.ldb);
        if (dma == D128x128k64r) return launch_bf16_dma_stats<128, 64, 4, 1, 3, true>(g, (hipStream_t)stream);
        if (dma == D64x64k64s4) return launch_bf16_dma_stats<64, 64, 2, 2, 4>(g, (hipStream_t)stream);
        if (stats_256x128(dma, g.M, g.N, BB_NT)) return launch_bf16_dma_stats<256, 128, 4, 2>(g, (hipStream_t)stream);
        return launch_bf16_dma_stats<128, 64, 4, 1>(g, (hipStream_t)stream);
    }
    GemmArgs g;
    int64_t batches;
    bool ta, tb;
    int rc = fill_args(d, g, batches, ta, tb);
    if (rc) return rc;
    if (d->M == 0 || d->N == 0) return BB_OK;
    hipStream_t st = (hipStream_t)stream;
    if (d->colsum_out) {
        if (colsum_fusable(d, batches)) g.colsum = d->colsum_out;
        else if ((rc = colsum_standalone(d, stream)) != BB_OK) return rc;
    }
    if (d->dtype == BB_BF16) {
        if (!ta && !tb) return dispatch_bf16<false, false>(g, (int)batches, st);
        if (!ta && tb) return dispatch_bf16<false, true>(g, (int)batches, st);
        return dispatch_bf16<true, true>(g, (int)batches, st);
    }
    if (const PiecesTile tile = pick_pieces(d, 1)) return launch_pieces(g, d->layout, tile, st);
    if (!ta && !tb) return dispatch_f32<false, false>(g, (int)batches, st);
    if (!ta && tb) return dispatch_f32<false, true>(g, (int)batches, st);
    return dispatch_f32<true, true>(g, (int)batches, st);
}

template <int BM, int BN, int WM, int WN, bool BKM, int STAGES, bool STATS = false>
static int launch_conv3x3(GemmArgs& g, const ConvArgs& cv, hipStream_t st) {
    constexpr int smem = STAGES * (BM + BN) * 64 * 2;
    auto kern = conv3x3_bf16_igemm_kernel<BM, BN, WM, WN, BKM, STAGES, STATS>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n), dim3(WM * WN * 64), smem, st, g, cv);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

template <int BM, int BN, int WM, int WN, int STAGES>
static int launch_conv3x3_bnbwd(GemmArgs& g, const ConvArgs& cv, const BnBwdArgs& bn, hipStream_t st) {
    constexpr int smem = STAGES * (BM + BN) * 64 * 2;
    auto kern = conv3x3_bf16_igemm_bnbwd_kernel<BM, BN, WM, WN, STAGES>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n), dim3(WM * WN * 64), smem, st, g, cv, bn);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
// one 64x64 tile per CU at most: as pick_dma_tile
static bool conv_small_tiles(int M, int N) { return (int64_t)((M + 63) / 64) * ((N + 63) / 64) <= 256; }

extern "C" int bb_conv3x3_supported(int dtype, int mode, int n, int h, int w, int cin, int cout) {
    const int64_t rows = (int64_t)n * h * w;
    const int gathered = mode == BB_CONV_DGRAD ? cout : cin, produced = mode == BB_CONV_DGRAD ? cin : cout;
    return dtype == BB_BF16 && (mode == BB_CONV_FWD || mode == BB_CONV_DGRAD) && n > 0 && h > 0 && w > 0 &&
           rows >= 128 && rows < (1ll << 31) && gathered >= 64 && gathered % 64 == 0 && produced % 8 == 0 &&
           produced >= 64;
}

extern "C" int bb_conv3x3(int dtype, int mode, int n, int h, int w, int cin, int cout, const void* src, const void* weight,
                          void* dst, float* strip_stats, void* stream) {
    BB_REQUIRE(src && weight && dst, "bb_conv3x3: null operand");
    BB_REQUIRE(!strip_stats || (mode == BB_CONV_FWD && ((uintptr_t)strip_stats % 16) == 0),
               "bb_conv3x3: strip_stats goes with BB_CONV_FWD only and must be 16-byte aligned");
    BB_REQUIRE(bb_conv3x3_supported(dtype, mode, n, h, w, cin, cout),
               "bb_conv3x3: unsupported problem (bf16, >= 128 pixels, gathered channels a multiple of 64, produced channels "
               "a multiple of 8 and >= 64): dtype %d mode %d n %d h %d w %d cin %d cout %d",
               dtype, mode, n, h, w, cin, cout);
    BB_REQUIRE(((uintptr_t)src % 16) == 0 && ((uintptr_t)weight % 16) == 0 && ((uintptr_t)dst % 16) == 0,
               "bb_conv3x3: operands must be 16-byte aligned");
    const bool dgrad = mode == BB_CONV_DGRAD;
    GemmArgs g = {};
    ConvArgs cv = {};
    g.M = n * h * w;
    g.N = dgrad ? cin : cout;
    g.K = 9 * (dgrad ? cout : cin);
    g.nb2 = 1;
    g.A = src;
    g.C = dst;
    g.lda = dgrad ? cout : cin;
    g.ldc = g.ldaux = g.N;
    g.alpha = 1.f;
    g.epilogue = BB_EPI_NONE;
    cv.h = h; cv.w = w; cv.c = dgrad ? cout : cin;
    hipStream_t st = (hipStream_t)stream;
    const bool small = conv_small_tiles(g.M, g.N);
    if (!dgrad) {
        // B = the weight as it lies: [cout, 9 * cin], k-contiguous
        g.B = weight;
        g.ldb = 9 * (int64_t)cin;
        if (strip_stats) {
            g.strip_stats = strip_stats;
            if (small) return launch_conv3x3<64, 64, 2, 2, false, 4, true>(g, cv, st);
            return launch_conv3x3<128, 64, 4, 2, false, 3, true>(g, cv, st);
        }
        if (small) return launch_conv3x3<64, 64, 2, 2, false, 4>(g, cv, st);
        // eight waves on a 128x64 tile (32x32 per wave): with one block per CU, two waves per SIMD hide each other's
        // LDS and barrier waits (four waves: 21.6 us, eight: 19.4 us at 6272 pixels, 256 channels)
        return launch_conv3x3<128, 64, 4, 2, false, 3>(g, cv, st);
    }
    // B[k = t * cout + o, n = i] = weight[o, 8 - t, i]: k-major with row stride 9 * cin, starting at tap 8; after
    // the cout / 64 k-tiles of a tap the rows go back to o = 0 and one tap down
    g.B = (const bf16*)weight + 8 * (int64_t)cin;
    g.ldb = 9 * (int64_t)cin;
    cv.b_every = cout / 64;
    cv.b_wrap = -(int64_t)cout * g.ldb - cin;
    if (small) return launch_conv3x3<64, 64, 2, 2, true, 4>(g, cv, st);
    return launch_conv3x3<64, 128, 2, 4, true, 3>(g, cv, st);
}

extern "C" int bb_conv3x3_dgrad_bn(int dtype, int n, int h, int w, int cin, int cout, const void* src, const void* weight, void* dst,
                                   const void* relu_out, const bb_bn_bwd_stats* bn, void* stream) {
    BB_REQUIRE(src && weight && dst, "bb_conv3x3_dgrad_bn: null operand");
    BB_REQUIRE(bb_conv3x3_supported(dtype, BB_CONV_DGRAD, n, h, w, cin, cout),
               "bb_conv3x3_dgrad_bn: unsupported problem (see bb_conv3x3): dtype %d n %d h %d w %d cin %d cout %d", dtype, n, h, w, cin, cout);
    BB_REQUIRE(((uintptr_t)src % 16) == 0 && ((uintptr_t)weight % 16) == 0 && ((uintptr_t)dst % 16) == 0 && ((uintptr_t)relu_out % 16) == 0,
               "bb_conv3x3_dgrad_bn: operands must be 16-byte aligned");
    int rc = check_bn_bwd_stats("bb_conv3x3_dgrad_bn", bn);
    if (rc) return rc;
    GemmArgs g = {};
    ConvArgs cv = {};
    g.M = n * h * w;
    g.N = cin;
    g.K = 9 * cout;
    g.nb2 = 1;
    g.A = src;
    g.C = dst;
    g.lda = cout;
    g.ldc = g.ldaux = g.N;
    g.alpha = 1.f;
    g.epilogue = relu_out ? BB_EPI_MUL_POS : BB_EPI_NONE;
    g.aux_in = relu_out;
    cv.h = h; cv.w = w; cv.c = cout;
    // the flipped filter read in place, as in bb_conv3x3
    g.B = (const bf16*)weight + 8 * (int64_t)cin;
    g.ldb = 9 * (int64_t)cin;
    cv.b_every = cout / 64;
    cv.b_wrap = -(int64_t)cout * g.ldb - cin;
    const BnBwdArgs b = {bn->x, bn->mean, bn->rstd, bn->strips};
    if (conv_small_tiles(g.M, g.N)) return launch_conv3x3_bnbwd<64, 64, 2, 2, 4>(g, cv, b, (hipStream_t)stream);
    return launch_conv3x3_bnbwd<64, 128, 2, 4, 3>(g, cv, b, (hipStream_t)stream);
}

template <bool TA, bool TB, bool CONVB = false> static int launch_grouped(GroupedArgs& G, hipStream_t st) {
    constexpr int BM = 128, BN = 128, STAGES = 3;
    constexpr int smem = STAGES * (BM + BN) * 32 * 2;
    int blocks = 0;
    for (int i = 0; i < G.count; ++i) {
        GemmArgs& g = G.p[i];
        g.tiles_m = (g.M + BM - 1) / BM;
        g.tiles_n = (g.N + BN - 1) / BN;
        G.first_block[i] = blocks;
        blocks += g.tiles_m * g.tiles_n;
    }
    G.first_block[G.count] = blocks;
    auto kern = gemm_bf16_dma_grouped_kernel<BM, BN, 2, 2, TA, TB, true, STAGES, CONVB, !TA && !TB>;
    // (the waves of a block in lock step, hidden size 1024 (x 4 in the feed-forward) and 8192 rows, in step / free: forward products 406 / 411 us,
    // input gradients 384 / 362)
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    bb_launch(kern, dim3(G.ride.blocks + blocks), dim3(256), smem, st, G);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// Weight gradients on the tiles of gemm_m16.h: plain fp32 sums over contractions from kM16WgradRows rows on (below, what such a launch does is
// read and write C, which three blocks a CU of 128x128 tiles do sooner: hidden size 1024 (x 4 in the feed-forward), 128x128 tiles of
// gemm_bf16_dma_grouped_kernel / the better of these, us: 128 rows 22.7 / 25.0, 256 26.8 / 27.5, 512 33.5 / 32.5, 1024 43.7 / 42.8).  The tile -- or that
// kernel -- by an estimate: outputs, rounds, K steps of the fullest CU and of the share of the CUs that have a tile.  Fitted to 660 layers of 600 to
// 16000 rows, 384 to 2048 wide (off by 4 to 6 %, 2-norm); of 595 from 768 rows on it leaves two more than 3 % slower than that kernel (3.2), where rounds alone,
// without it among the choices, left 37, up to 14 %.  us (the one taken marked; - what rounds alone took):
//     hidden size, rows    before, three a CU    256x256    192x256    128x256    128x128, two a CU
//     1024      8192             229               184*       280        215         204
//     1024      4096             119               101*       154        120         110
//     1600      4096             282               301        254*       295         265
//      960      8200             219               182        161*       215         207
//      768     16384             285               326        256        223*        242
//      768      8192             148               174        135        113*        121
//      768      2043              46                59         47         40*         40
//      640      3000              58                78         61         48*         51
//     1408       917              88*               99-       107         96          86     (in the cache 70 / 85 / 94 / 93 / 79)
//     1472 (x2) 1031              76*               96         85-        83          77
//     1184      1285              86*              104         93-        91          88
//     1792       976             141               151-       153        139*        141
// Tried: 160-wide tiles (rows of 320 bytes, no whole lines: 1600 284); 32-wide k-tiles in rings of four and five (1024 8192 195, 202 against 187).
constexpr int kM16WgradRows = 768;
enum WgradTile { WG_NONE = 0, WG256x256, WG192x256, WG128x256, WG128x128 };
static WgradTile pick_wgrad_m16(const GroupedArgs& G) {
    static const struct {
        WgradTile tile;
        int bm, bn, blocks, sum_columns;                    // blocks a CU
        double base, outputs, round, share, full, step[4];  // us; us per 10^6 outputs, per round; per k: times the share, of a full CU, of one with so many blocks
    } tiles[] = {{WG_NONE, 128, 128, 3, 0, 7.2, 1.45, 2.0, 0.0087, 0.0126, {0, 0.0112, 0.0116, 0.0160}},
                 {WG256x256, 256, 256, 1, m16_sum_columns(8, 4), 9.2, 1.32, 8.3, -0.0005, 0.0215, {0, 0.0215}},
                 {WG192x256, 192, 256, 1, m16_sum_columns(6, 4), 8.0, 1.26, 6.1, 0.0002, 0.0181, {0, 0.0181}},
                 {WG128x256, 128, 256, 1, m16_sum_columns(4, 4), 7.2, 0.96, 6.0, 0.0031, 0.0098, {0, 0.0098}},
                 {WG128x128, 128, 128, 2, m16_sum_columns(4, 2), 5.6, 1.14, 3.6, 0.0054, 0.0090, {0, 0.0107, 0.0112}}};
    int kmax = 0;
    double outputs = 0.0;
    for (int i = 0; i < G.count; ++i) {
        const GemmArgs& g = G.p[i];
        if (!g.c_f32 || g.bias || g.epilogue != BB_EPI_NONE || g.K < kM16WgradRows || g.lda >= kDmaMaxLd || g.ldb >= kDmaMaxLd || g.conv_c != 0) return WG_NONE;
        kmax = g.K > kmax ? g.K : kmax;
        outputs += 1e-6 * g.M * g.N;
    }
    const int k = (kmax + 63) / 64 * 64;
    WgradTile best = WG_NONE;
    double least = 0.0;
    for (const auto& t : tiles) {
        int64_t n = 0;
        bool fits = true;
        for (int i = 0; i < G.count; ++i) {
            const GemmArgs& g = G.p[i];
            const int columns = (g.N + t.bn - 1) / t.bn;
            fits = fits && (!g.colsum || columns >= t.sum_columns);
            n += (int64_t)((g.M + t.bm - 1) / t.bm) * columns;
        }
        const int64_t slots = (int64_t)t.blocks * kCUs, full = (n - 1) / slots, most = (n - slots * full + kCUs - 1) / kCUs;
        const double us = t.base + t.outputs * outputs + t.round * (full + 1) + (full * t.full + t.step[most] + t.share * n / slots) * k;
        // (few k-tiles and all of it in the last-level cache: that kernel is another tenth faster)
        if (t.tile == WG_NONE) least = (k < 2048 ? 0.95 : 1.0) * us;
        else if (fits && us < least) best = t.tile, least = us;
    }
    return best;
}
template <int TM, int TN, int WM, int WN, int STAGES> static int launch_wgrad_m16(GroupedArgs& G, hipStream_t st) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16, smem = STAGES * (BM + BN) * 128;
    static_assert(kM16WgradRows > STAGES * 64, "the ring is filled before the last k-tile");
    auto kern = wgrad_m16_grouped_kernel<TM, TN, WM, WN, STAGES>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    int blocks = 0;
    for (int i = 0; i < G.count; ++i) {
        GemmArgs& g = G.p[i];
        g.tiles_m = (g.M + BM - 1) / BM;
        g.tiles_n = (g.N + BN - 1) / BN;
        G.first_block[i] = blocks;
        blocks += g.tiles_m * g.tiles_n;
    }
    G.first_block[G.count] = blocks;
    bb_launch(kern, dim3(G.ride.blocks + blocks), dim3(WM * WN * 64), smem, st, G);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// A layer's weight gradients with up to four 64x64 tiles per CU, i.e. at most one 128x128 tile: that one is a chain of
// k-tiles nobody overlaps.  Eight waves a tile while there is one tile per CU, four (two blocks a CU) above.  128x128 tiles /
// 64x64 tiles (us), rows x hidden (x 4 in the feed-forward): 300x256 12.1 / 7.3, 3378x192 61.6 / 16.9, 8000x192 132 / 31,
// 1050x512 27.4 / 22.3, 3001x320 57.6 / 26.6; 2048x768 (1728 tiles) 48 / 56.
constexpr int64_t kGroupedWaveTiles = 1024;
template <int KW, int BK, int NST> static int launch_grouped_wave(GroupedArgs& G, bool conv, hipStream_t st) {
    auto kern = conv ? gemm_bf16_wave_grouped_kernel<true, true, KW, BK, NST, true> : gemm_bf16_wave_grouped_kernel<true, true, KW, BK, NST>;
    constexpr int smem = wave_gemm_lds(KW, BK, NST);
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    int blocks = 0;
    for (int i = 0; i < G.count; ++i) {
        GemmArgs& g = G.p[i];
        g.tiles_m = (g.M + 63) / 64;
        g.tiles_n = (g.N + 63) / 64;
        G.first_block[i] = blocks;
        blocks += g.tiles_m * g.tiles_n;
    }
    G.first_block[G.count] = blocks;
    bb_launch(kern, dim3(G.ride.blocks + blocks), dim3(KW * 64), smem, st, G);
    BB_LAUNCH_CHECK();
    return BB_OK;
}

// The bias gradients that ride on fp32 weight gradients: one pair of launches for all of them where their workspaces do not
// overlap, else a pair each.
static int colsum_f32(const bb_gemm_desc* descs, int count, void* stream) {
    BbColsumGroup C;
    C.count = 0;
    bool apart = true;
    for (int i = 0; i < count; ++i) {
        const bb_gemm_desc& d = descs[i];
        if (!d.colsum_out) continue;
        BB_REQUIRE(d.colsum_ws, "bb_gemm_grouped: colsum_out on this problem needs colsum_ws");
        const float *lo = d.colsum_ws, *hi = lo + bb_colsum_workspace(d.M);
        for (int j = 0; j < C.count; ++j) apart = apart && (hi <= C.partial[j] || C.partial[j] + bb_colsum_workspace(C.cols[j]) <= lo);
        C.x[C.count] = (const float*)d.A; C.partial[C.count] = d.colsum_ws; C.out[C.count] = d.colsum_out;
        C.ldx[C.count] = d.lda; C.rows[C.count] = d.K; C.cols[C.count] = d.M;
        ++C.count;
    }
    if (C.count == 0) return BB_OK;
    if (apart) return bb_colsum_acc_grouped(C, (hipStream_t)stream);
    for (int i = 0; i < count; ++i) {
        int rc = descs[i].colsum_out ? colsum_standalone(&descs[i], stream) : BB_OK;
        if (rc) return rc;
    }
    return BB_OK;
}

// whether the grouped DMA kernel takes the problem: it masks the contraction's end for weight gradients only
static bool shared_launch_dma(const bb_gemm_desc& d) {
    const DmaTile t = narrow_or_wide(pick_dma_tile(d.M, d.N, d.K, 1, d.layout), d.layout, d.lda, d.ldb);
    return t != D_NONE && t != D128x128k64r;
}

extern "C" int bb_gemm_grouped_sums(const bb_gemm_desc* descs, int count, const bb_partial_sums* sums, int nsums, void* stream) {
    BB_REQUIRE(count >= 0 && (descs || count == 0), "bb_gemm_grouped: bad arguments");
    hipStream_t st = (hipStream_t)stream;
    PartialSums ride;
    int ride_rc = bb_partial_sums_args("bb_gemm_grouped_sums", sums, nsums, ride);
    if (ride_rc) return ride_rc;
    if (!bb_partial_sums_apart(sums, nsums)) {     // into the same memory: one after the other, in launches of their own
        ride_rc = bb_partial_sums_acc(sums, nsums, stream);
        return ride_rc ? ride_rc : bb_gemm_grouped_sums(descs, count, nullptr, 0, stream);
    }
    // one launch when every problem is an unbatched bf16 problem of one layout that the DMA
    // kernel accepts; otherwise the problems run one after the other (same results)
    bool has_conv = false;
    for (int i = 0; i < count; ++i) has_conv = has_conv || descs[i].conv_c != 0;
    bool fuse = count >= (has_conv ? 1 : 2) && count <= GROUP_MAX, dma = true, wave = count > 0 && descs[0].layout == BB_TN;
    int64_t tiles = 0;
    for (int i = 0; i < count && fuse; ++i) {
        const bb_gemm_desc& d = descs[i];
        // the grouped kernels are built without dropout decisions in their epilogue: such a problem runs by itself
        dma = dma && shared_launch_dma(d) && d.conv_c % 128 == 0;
        wave = wave && pick_wave(d.M, d.N, d.K, 1, d.layout, D_NONE) != W_NONE;
        fuse = d.dtype == BB_BF16 && d.layout == descs[0].layout && d.nb1 <= 1 && d.nb2 <= 1 && d.M > 0 && d.N > 0 &&
               d.dropout_p == 0.f && (dma || wave);
        tiles += (int64_t)((d.M + 63) / 64) * ((d.N + 63) / 64);
    }
    // weight gradients of few tiles: 64x64 tiles, the contraction dealt to the waves (see kGroupedWaveTiles)
    wave = wave && (!dma || tiles <= (count > 1 ? kGroupedWaveTiles : 256));   // alone: as bb_gemm takes it
    if (!fuse && count >= 2 && pick_pieces(descs, count)) {
        GroupedArgs G;
        G.count = count;
        G.ride = ride;
        for (int i = 0; i < count; ++i) {
            int64_t batches;
            bool ta, tb;
            int rc = fill_args(&descs[i], G.p[i], batches, ta, tb);
            if (rc) return rc;
        }
        const int rc = colsum_f32(descs, count, stream);
        return rc ? rc : launch_pieces_grouped(G, st);
    }
    // fp32: unbatched problems of one layout share a launch where one kernel takes them all (weight gradients of both kinds:
    // the 64x64 tiles)
    bool fuse32 = !fuse && !has_conv && count >= 2 && count <= GROUP_MAX;
    int few = 0;
    for (int i = 0; i < count && fuse32; ++i) {
        const bb_gemm_desc& d = descs[i];
        const bool w = pick_f32_wave(d.M, d.N, d.K, 1, d.layout);
        few += w;
        fuse32 = d.dtype == BB_F32 && d.layout == descs[0].layout && d.nb1 <= 1 && d.nb2 <= 1 && d.M > 0 && d.N > 0 && d.dropout_p == 0.f &&
                 !f32_wide(d.lda, d.ldb) &&
                 (w || !pick_f32_split(d.M, d.N, d.K, 1, d.layout));
    }
    const bool waves = few == count;
    fuse32 = fuse32 && (waves || few == 0 || descs[0].layout == BB_TN);
    if (fuse32) {
        GroupedArgs G;
        G.count = count;
        G.ride = ride;
        int64_t tiles64 = 0;
        for (int i = 0; i < count; ++i) tiles64 += (int64_t)((descs[i].M + 63) / 64) * ((descs[i].N + 63) / 64);
        // weight gradients: on quarter tiles (the bits of 64x64 ones) by the tiles of all of them
        const bool quarter = !waves && descs[0].layout == BB_TN && tiles64 <= kF32QuarterTiles;
        const int tile = waves || quarter ? 32 : 64;
        int blocks = 0;
        for (int i = 0; i < count; ++i) {
            int64_t batches;
            bool ta, tb;
            int rc = fill_args(&descs[i], G.p[i], batches, ta, tb);
            if (rc) return rc;
            G.p[i].tiles_m = (G.p[i].M + tile - 1) / tile;
            G.p[i].tiles_n = (G.p[i].N + tile - 1) / tile;
            G.first_block[i] = blocks;
            blocks += G.p[i].tiles_m * G.p[i].tiles_n;
        }
        G.first_block[count] = blocks;
        int rc = colsum_f32(descs, count, stream);
        if (rc) return rc;
        const int layout = descs[0].layout;
        const auto kern = quarter            ? gemm_f32_quarter_grouped_kernel
                          : layout == BB_NT ? gemm_f32_grouped_kernel<false, false>
                          : layout == BB_NN ? waves ? gemm_f32_wave_grouped_kernel<false, true> : gemm_f32_grouped_kernel<false, true>
                                            : waves ? gemm_f32_wave_grouped_kernel<true, true> : gemm_f32_grouped_kernel<true, true>;
        bb_launch(kern, dim3(G.ride.blocks + blocks), dim3(256), waves ? kF32WaveLds : quarter ? kF32QuarterLds : f32_gemm_lds(64), st, G);
        BB_LAUNCH_CHECK();
        return BB_OK;
    }
    // a patch-matrix B exists only inside the grouped kernels: no one-by-one route for it
    BB_REQUIRE(fuse || !has_conv, "bb_gemm_grouped: a problem with a patch-matrix B must share a launch of unbatched bf16 BB_TN problems");
    if (!fuse) {
        int rc = bb_partial_sums_acc(sums, nsums, stream);
        if (rc) return rc;
        for (int i = 0; i < count; ++i) {
            rc = bb_gemm(&descs[i], stream);
            if (rc) return rc;
        }
        return BB_OK;
    }
    GroupedArgs G;
    G.count = count;
    G.ride = ride;
    for (int i = 0; i < count; ++i) {
        int64_t batches;
        bool ta, tb;
        int rc = fill_args(&descs[i], G.p[i], batches, ta, tb);
        if (rc) return rc;
        if (descs[i].colsum_out) G.p[i].colsum = descs[i].colsum_out;  // both grouped kernels leave the sums
    }
    const int layout = descs[0].layout;
    if (wave && tiles <= 256) return launch_grouped_wave<8, 32, 2>(G, has_conv, st);
    if (wave) return launch_grouped_wave<4, 32, 2>(G, has_conv, st);
    if (layout == BB_NT) return launch_grouped<false, false>(G, st);
    if (layout == BB_NN) return launch_grouped<false, true>(G, st);
    if (has_conv) return launch_grouped<true, true, true>(G, st);
    switch (pick_wgrad_m16(G)) {
        case WG256x256: return launch_wgrad_m16<8, 4, 2, 4, 2>(G, st);
        case WG192x256: return launch_wgrad_m16<6, 4, 2, 4, 2>(G, st);
        case WG128x256: return launch_wgrad_m16<4, 4, 2, 4, 3>(G, st);
        case WG128x128: return launch_wgrad_m16<4, 4, 2, 2, 2>(G, st);
        default: return launch_grouped<true, true>(G, st);
    }
}
extern "C" int bb_gemm_grouped(const bb_gemm_desc* descs, int count, void* stream) {
    return bb_gemm_grouped_sums(descs, count, nullptr, 0, stream);
}

// =========================================================================================
// Grouped GEMMs with few output tiles and a long contraction (the weight gradients of a ResNet
// bottleneck: 68 tiles of 128x128 over K = 6272 rows): the contraction is cut into `splits`
// chunks, each chunk of each problem becomes a problem of its own that writes an fp32 partial
// product into the caller's workspace, and a second kernel adds the partials to C in chunk order.
// =========================================================================================
constexpr int SPLITK_MAX = 8;

// every problem of the group in one launch: blockIdx.y = problem
struct SplitkReduceArgs {
    const float* ws[GROUP_MAX];
    float* C[GROUP_MAX];
    int64_t ldc[GROUP_MAX];
    int M[GROUP_MAX], N[GROUP_MAX], accumulate[GROUP_MAX];
    int splits;
};
template <> struct BbPointersAt<SplitkReduceArgs> : BbPointerRun<2 * GROUP_MAX> {};   // ws, C
static_assert(offsetof(SplitkReduceArgs, ldc) == 2 * GROUP_MAX * sizeof(void*), "BbPointersAt<SplitkReduceArgs>");
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const SplitkReduceArgs a) {
    const int pi = blockIdx.y;
    const int M = a.M[pi], N = a.N[pi], splits = a.splits, accumulate = a.accumulate[pi];
    const float* __restrict__ ws = a.ws[pi];
    float* __restrict__ C = a.C[pi];
    const int64_t ldc = a.ldc[pi], part = (int64_t)M * N;
    const int64_t nvec = part / 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * 256) {
        const int64_t e = i * 4;
        const int m = (int)(e / N), n = (int)(e % N);
        float* c = C + (int64_t)m * ldc + n;
        f32x4 acc = accumulate ? *(const f32x4*)c : f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 v[SPLITK_MAX];
#pragma unroll
        for (int p = 0; p < SPLITK_MAX; ++p)
            if (p < splits) v[p] = *(const f32x4*)(ws + p * part + e);
#pragma unroll
        for (int p = 0; p < SPLITK_MAX; ++p)
            if (p < splits) acc += v[p];
        *(f32x4*)c = acc;
    }
}

// chunks of the contraction: 0 or 1 = run the group whole
static int pick_splits(const bb_gemm_desc* descs, int count) {
    if (count < 1 || count > GROUP_MAX) return 0;
    int64_t tiles = 0, tiles128 = 0;
    int kmin = 1 << 30;
    for (int i = 0; i < count; ++i) {
        const bb_gemm_desc& d = descs[i];
        if (d.dtype != BB_BF16 || d.c_dtype != BB_F32 || d.layout != descs[0].layout || d.nb1 > 1 || d.nb2 > 1 || d.M <= 0 ||
            d.N <= 0 || d.colsum_out || d.bias || d.epilogue != BB_EPI_NONE || d.alpha != 1.0f || d.N % 4 != 0 || d.dropout_p != 0.f ||
            (!shared_launch_dma(d) && d.layout != BB_TN))
            return 0;
        tiles += (int64_t)((d.M + 63) / 64) * ((d.N + 63) / 64);
        tiles128 += (int64_t)((d.M + 127) / 128) * ((d.N + 127) / 128);
        kmin = d.K < kmin ? d.K : kmin;
    }
    // Few tiles: 64x64 ones with eight waves, and chunks while those leave half the CUs idle (at least 1024 rows a chunk, four
    // slices a wave).  More tiles: whole on 64x64 tiles while the contraction is short, else chunks of 128x128 tiles for two
    // blocks per CU -- with one, a CU's four waves have nobody to hide their load and barrier waits behind.  Weight gradients
    // of a ResNet block, 128x128 tiles in their best split / this rule (us with the reduction), rows, middle channels: 12544,
    // 128 52 / 23; 12544, 64 (patch matrix) / 17; 900, 128 14.6 / 8.7; 3136, 256 28.8 / 25.9; 648, 256 19.8 / 11.0;
    // 6272, 256 40 on five chunks of 128x128 tiles, 44 whole.
    int splits, least = 1024;
    if (tiles <= 256) splits = tiles > 128 ? 1 : (int)(384 / tiles);
    else if (tiles <= kGroupedWaveTiles && kmin <= 4096) return 1;
    else {
        splits = (int)(256 * 2 / tiles128);
        least = 512;
    }
    if (splits > SPLITK_MAX) splits = SPLITK_MAX;
    if (splits > GROUP_MAX / count) splits = GROUP_MAX / count;
    while (splits > 1 && kmin / splits < least) --splits;
    return splits;
}

extern "C" int64_t bb_gemm_splitk_workspace(const bb_gemm_desc* descs, int count) {
    int64_t n = 0;
    for (int i = 0; descs && i < count; ++i) n += (int64_t)descs[i].M * descs[i].N;
    return n * SPLITK_MAX * (int64_t)sizeof(float);
}

extern "C" int bb_gemm_grouped_splitk(const bb_gemm_desc* descs, int count, void* workspace, int64_t workspace_bytes,
                                      void* stream) {
    BB_REQUIRE(count >= 0 && (descs || count == 0), "bb_gemm_grouped_splitk: bad arguments");
    const int splits = pick_splits(descs, count);
    if (splits <= 1) return bb_gemm_grouped(descs, count, stream);
    int64_t need = 0;
    for (int i = 0; i < count; ++i) need += (int64_t)descs[i].M * descs[i].N * splits * (int64_t)sizeof(float);
    BB_REQUIRE(workspace && workspace_bytes >= need && ((uintptr_t)workspace % 16) == 0,
               "bb_gemm_grouped_splitk: workspace of %lld bytes needed (16-byte aligned), got %lld", (long long)need,
               (long long)workspace_bytes);
    bb_gemm_desc sub[GROUP_MAX];
    float* ws = (float*)workspace;
    int ns = 0;
    for (int i = 0; i < count; ++i) {
        const bb_gemm_desc& d = descs[i];
        // chunk boundaries on multiples of 32 rows of the contraction
        const int kt = d.K / 32, per = kt / splits, extra = kt % splits;
        int k0 = 0;
        for (int p = 0; p < splits; ++p) {
            int kc = (per + (p < extra ? 1 : 0)) * 32;
            if (p == splits - 1) kc = d.K - k0;
            bb_gemm_desc& t = sub[ns++];
            t = d;
            t.K = kc;
            // A advances along its contraction index: rows for TN ([K, M]), columns otherwise ([M, K])
            t.A = (const char*)d.A + (d.layout == BB_TN ? (int64_t)k0 * d.lda : (int64_t)k0) * 2;
            // B: [N, K] for NT, [K, N] for NN and TN
            if (d.conv_c != 0) t.conv_row0 = d.conv_row0 + k0;   // the tensor stays put, the chunk starts k0 pixels in
            else t.B = (const char*)d.B + (d.layout == BB_NT ? (int64_t)k0 : (int64_t)k0 * d.ldb) * 2;
            t.C = ws + (int64_t)p * d.M * d.N;
            t.ldc = d.N;
            t.accumulate = 0;
            k0 += kc;
        }
        ws += (int64_t)splits * d.M * d.N;
    }
    int rc = bb_gemm_grouped(sub, ns, stream);
    if (rc) return rc;
    SplitkReduceArgs ra;
    ra.splits = splits;
    ws = (float*)workspace;
    int64_t most = 0;
    for (int i = 0; i < count; ++i) {
        const bb_gemm_desc& d = descs[i];
        const int64_t part = (int64_t)d.M * d.N;
        ra.ws[i] = ws; ra.C[i] = (float*)d.C; ra.ldc[i] = d.ldc;
        ra.M[i] = d.M; ra.N[i] = d.N; ra.accumulate[i] = d.accumulate;
        most = part / 4 > most ? part / 4 : most;
        ws += (int64_t)splits * part;
    }
    const unsigned bx = (unsigned)((most + 255) / 256 > 1024 ? 1024 : (most + 255) / 256);
    bb_launch(splitk_reduce_kernel, dim3(bx, (unsigned)count), dim3(256), 0, (hipStream_t)stream, ra);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
