// bf16 weight gradients, and products whose contraction is no multiple of 32, that do not fill the chip: 64x64 tiles whose
// contraction is dealt to the KW waves of a block.
#pragma once
#include "gemm_kernels.h"

// What bounds such a problem is not a rate but a chain: k-tile after k-tile, each a wait for its loads, a barrier, LDS
// reads and a few matrix instructions (0.9 us per 32 rows on a 128x128 tile with one block per CU), then an epilogue of
// dependent round trips.  Here a wave owns whole 32-wide slices of the contraction (wave w: slices w, w + KW, ...) of the block's full
// 64x64 tile: it loads them into a ring of its own, waits for nobody -- no barrier in the loop --, and the chain is KW
// times shorter.  The KW partial tiles meet in LDS once and are added in wave order; each lane then finishes one row
// segment of eight columns (KW = 8: the whole epilogue is one pass, its operands fetched before the main loop).
// No operand byte is loaded twice by a block (the slices are disjoint), so this costs no traffic against any other
// 64x64 tiling; against larger tiles it costs loads, which is why it is for problems of few tiles.  A sum is added up in
// another order than in the DMA kernels; forward products, whose last bits decide ReLUs, stay with those (64x64 tiles there)
// where K % 32 == 0.
// The contraction may have any length: slices past its end read a line of zeros.
// 64 rows x BK k of one operand, loaded by one wave.  CONV (k-major): the rows are columns of the 3x3 patch matrix of an NHWC
// tensor, k its pixels; a 64-wide tile lies inside one tap (the channel count is a multiple of 64), a lane reads the channels
// of the pixel `tap` away from its own, or zeros where that leaves the image.
template <bool KM, int BK, bool CONV = false> struct SliceOperand {
    static_assert(KM || !CONV, "the gathered operand is k-major");
    static constexpr int BYTES = 64 * BK * 2, ROUNDS = BYTES / 1024;
    const bf16* src[ROUNDS];
    int64_t step;      // elements per slice of this wave
    int k_lane;        // k of the lane's 16 bytes inside a slice (round 0)
    const bf16* zero;
    int py[CONV ? ROUNDS : 1], px[CONV ? ROUNDS : 1], tdy, tdx, dpy, dpx, h, w;   // CONV: image coordinates of the lane's pixels
    __device__ __forceinline__ void init_conv(const GemmArgs& g, const bf16* base, int col0, int lane, int slice0, int stride) {
        h = g.conv_h; w = g.conv_w;
        const int t = col0 / g.conv_c, ci0 = col0 - t * g.conv_c;
        tdy = t / 3 - 1; tdx = t % 3 - 1;
        dpy = stride * BK / w % h; dpx = stride * BK % w;
        k_lane = lane >> 3;
        const int c = (lane & 7) ^ km_swizzle<64>(lane >> 3);
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int p = g.conv_row0 + slice0 * BK + i * 8 + (lane >> 3), pix = p % (h * w);
            py[i] = pix / w;
            px[i] = pix - py[i] * w;
            src[i] = base + ((int64_t)p + tdy * w + tdx) * g.conv_c + ci0 + c * 8;
        }
        step = (int64_t)stride * BK * g.conv_c;
        zero = (const bf16*)(bb_zero_line + (lane & 7) * 16);
    }
    __device__ __forceinline__ void init(const bf16* base, int64_t ld, int row0, int rows, int lane, int slice0, int stride) {
        if constexpr (!KM) {
            // as DmaOperand: an instruction takes 8 rows x 128 bytes (BK 64) or 16 rows x 64 bytes (BK 32)
            constexpr int CPR = BK / 8, RPI = 64 / CPR;
            const int c = BK == 64 ? (lane & 7) ^ ((lane >> 4) & 3) : (lane & 3) ^ ((lane >> 4) & 3);
            k_lane = c * 8;
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) {
                const int r = i * RPI + lane / CPR;
                const int ci = BK == 64 ? (lane & 7) ^ ((r >> 1) & 7) : c;
                src[i] = base + (int64_t)min(row0 + r, rows - 1) * ld + slice0 * BK + ci * 8;
            }
            step = stride * BK;
        } else {
            k_lane = lane >> 3;
            const int c = (lane & 7) ^ km_swizzle<64>(lane >> 3);
            const int col = min(row0 + c * 8, rows - 8);
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) src[i] = base + ((int64_t)slice0 * BK + i * 8 + (lane >> 3)) * ld + col;
            step = stride * BK * ld;
        }
        zero = (const bf16*)(bb_zero_line + (lane & 7) * 16);
    }
    // `left`: contraction elements from the slice's start to the end (< BK: the last, ragged slice)
    __device__ __forceinline__ void issue(unsigned char* stage, int left) {
        if constexpr (CONV) {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) {
                const bool in = k_lane + i * 8 < left && (unsigned)(py[i] + tdy) < (unsigned)h && (unsigned)(px[i] + tdx) < (unsigned)w;
                dma16(in ? src[i] : zero, stage + i * 1024);
                px[i] += dpx;
                py[i] += dpy;
                if (px[i] >= w) {
                    px[i] -= w;
                    ++py[i];
                }
                if (py[i] >= h) py[i] -= h;   // dpy < h: at most one image further
            }
        } else if (left >= BK) {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) dma16(src[i], stage + i * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) {
                // k of the lane's bytes: with 64-wide slices the swizzle of odd row groups differs in its third bit
                const int k = KM ? k_lane + i * 8 : BK == 64 ? k_lane ^ ((i & 1) << 5) : k_lane;
                dma16(k < left ? src[i] : zero, stage + i * 1024);
            }
        }
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) src[i] += step;
    }
};

// NST stages a wave, column sums
constexpr int wave_gemm_lds(int kw, int bk, int nst) { return kw * nst * (2 * 64 * 2 * bk) + kw * 64 * 4; }

template <bool AKM, bool BKM, int KW, int BK, int NST, bool DROP, bool CONVB = false>
__device__ __forceinline__ void gemm_bf16_wave_body(const GemmArgs& g, const int tile_m, const int tile_n, const int batch_id) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = tile_m * 64, n0 = tile_n * 64;
    const int b1 = batch_id / g.nb2, b2 = batch_id % g.nb2;
    const bf16* A = (const bf16*)g.A + b1 * g.sA1 + b2 * g.sA2;
    const bf16* B = (const bf16*)g.B + b1 * g.sB1 + b2 * g.sB2;
    const int64_t coff = b1 * g.sC1 + b2 * g.sC2;

    constexpr int OP = 64 * BK * 2, STAGE = 2 * OP, RING = NST * STAGE;
    static_assert(RING >= 64 * 64 * 4, "a wave's partial tile takes the place of its ring");
    SliceOperand<AKM, BK> opa;
    SliceOperand<BKM, BK, CONVB> opb;
    opa.init(A, g.lda, m0, g.M, lane, wave, KW);
    if constexpr (CONVB) opb.init_conv(g, B, n0, lane, wave, KW);
    else opb.init(B, g.ldb, n0, g.N, lane, wave, KW);
    FragReader<64, 2, AKM, BK> fa;
    FragReader<64, 2, BKM, BK> fb;
    fa.init(0, lane);
    fb.init(0, lane);
    unsigned char* ring = smem + wave * RING;

    // what the epilogue reads beside the product, for the rows this lane will finish
    constexpr int PASSES = 8 / KW;
    const int prow = wave * 8 + (lane >> 3), pcol = (lane & 7) * 8, n = n0 + pcol;
    const bf16* opnd = epilogue_operand(g);
    u32x4 pre[PASSES], pre2[PASSES];
    f32x4 c_lo[PASSES], c_hi[PASSES];
    float b8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (g.bias && n < g.N) load_vec((const bf16*)g.bias + n, b8);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int m = m0 + p * (8 * KW) + prow;
        pre[p] = pre2[p] = u32x4{0u, 0u, 0u, 0u};
        c_lo[p] = c_hi[p] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (m < g.M && n < g.N) {
            if (opnd) pre[p] = *(const u32x4*)(opnd + coff + (int64_t)m * g.ldaux + n);
            if (g.epilogue == BB_EPI_MUL_POS && g.resid) pre2[p] = *(const u32x4*)((const bf16*)g.resid + coff + (int64_t)m * g.ldaux + n);
            if (g.accumulate) {
                c_lo[p] = *(const f32x4*)((const float*)g.C + coff + (int64_t)m * g.ldc + n);
                c_hi[p] = *(const f32x4*)((const float*)g.C + coff + (int64_t)m * g.ldc + n + 4);
            }
        }
    }

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const bool do_colsum = AKM && g.colsum != nullptr && tile_n == 0;
    float csum[2] = {0.f, 0.f};

    const int slices = (g.K + BK - 1) / BK;
    const int mine = wave < slices ? (slices - wave + KW - 1) / KW : 0;
    int left = g.K - wave * BK;      // from the next slice to issue
    auto issue = [&](int stage) {
        opa.issue(ring + stage * STAGE, left);
        opb.issue(ring + stage * STAGE + OP, left);
        left -= KW * BK;
    };
    if (mine > 0) issue(0);
    if (NST > 1 && mine > 1) issue(1);
    for (int s = 0; s < mine; ++s) {
        asm volatile("" ::: "memory");
        if (NST > 1 && s + 1 < mine) wait_vmcnt_lgkm0<2 * OP / 1024>();   // in-order completion: slice s has landed, slice s + 1 may be in flight
        else wait_vmcnt_lgkm0<0>();
        asm volatile("" ::: "memory");
        const unsigned char* st = ring + (NST > 1 ? s & 1 : 0) * STAGE;
        bf16x8 a[BK / 16][2], b[BK / 16][2];
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[ks][i] = fa.load(st, i, ks);
                b[ks][i] = fb.load(st + OP, i, ks);
            }
        // the stage is read before its next slice may overwrite it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (s + NST < mine) issue(NST > 1 ? s & 1 : 0);
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
            if constexpr (AKM) {
                if (do_colsum) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        float t = 0.f;
#pragma unroll
                        for (int e = 0; e < 8; ++e) t += (float)a[ks][i][e];
                        csum[i] += t;
                    }
                }
            }
        }
    }
    // partial tiles through LDS, [64][64] floats a wave in its own (drained) ring; 16-byte chunk c of row r at c ^ (r & 15)
    float* part = (float*)ring;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = j * 32 + (lane & 31);
                part[row * 64 + ((((col >> 2) ^ (row & 15)) << 2) | (col & 3))] = acc[i][j][r];
            }
    float* csums = (float*)(smem + KW * RING);
    if constexpr (AKM) {
        if (do_colsum) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float t = csum[i] + __shfl_xor(csum[i], 32, 64);
                if (lane < 32) csums[wave * 64 + i * 32 + lane] = t;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int row = p * (8 * KW) + prow, m = m0 + row;
        const int at0 = row * 64 + (((pcol >> 2) ^ (row & 15)) << 2), at1 = row * 64 + ((((pcol >> 2) + 1) ^ (row & 15)) << 2);
        f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < KW; ++w) {
            const float* q = (const float*)(smem + w * RING);
            lo += *(const f32x4*)(q + at0);
            hi += *(const f32x4*)(q + at1);
        }
        float v[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = lo[e] * g.alpha;
            v[4 + e] = hi[e] * g.alpha;
        }
        if (m < g.M && n < g.N)
            epilogue_vec8_at<DROP, true, true, true>(g, coff + (int64_t)m * g.ldc + n, coff + (int64_t)m * g.ldaux + n, m, n, v, b8,
                                                     pre[p], pre2[p], c_lo[p], c_hi[p]);
    }
    if constexpr (AKM) {
        if (do_colsum && threadIdx.x < 64) {
            const int m = m0 + threadIdx.x;
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < KW; ++w) t += csums[w * 64 + threadIdx.x];
            if (m < g.M) g.colsum[m] += t;
        }
    }
}

template <bool AKM, bool BKM, int KW, int BK, int NST, bool DROP>
__global__ __launch_bounds__(KW * 64) void gemm_bf16_wave_kernel(const GemmArgs g) {
    int tile_m, tile_n;
    tile_coords(blockIdx.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
    gemm_bf16_wave_body<AKM, BKM, KW, BK, NST, DROP>(g, tile_m, tile_n, blockIdx.z);
}
// several unbatched problems in one launch
// CONVB: some of them read B as the patch matrix of a 3x3 convolution
template <bool AKM, bool BKM, int KW, int BK, int NST, bool CONVB = false>
__global__ __launch_bounds__(KW * 64) void gemm_bf16_wave_grouped_kernel(const GroupedArgs G) {
    const int lid = grouped_place<KW>(G);
    if (lid < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && lid >= G.first_block[pi + 1]) ++pi;
    int tile_m, tile_n;
    panel_coords(lid - G.first_block[pi], G.p[pi].tiles_m, G.p[pi].tiles_n, tile_m, tile_n);
    if constexpr (CONVB) {
        if (G.p[pi].conv_c > 0) {
            gemm_bf16_wave_body<AKM, BKM, KW, BK, NST, false, true>(G.p[pi], tile_m, tile_n, 0);
            return;
        }
    }
    gemm_bf16_wave_body<AKM, BKM, KW, BK, NST, false>(G.p[pi], tile_m, tile_n, 0);
}
