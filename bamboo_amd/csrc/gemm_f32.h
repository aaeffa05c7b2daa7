// fp32 GEMM: v_mfma_f32_16x16x4_f32 on 64x64 tiles (four waves of 32x32), on 64x32 tiles whose contraction two groups of
// two waves share, or on quarters of a 64x64 tile; v_mfma_f32_32x32x2_f32 on 32x32 tiles whose contraction four waves share.
#pragma once
#include "gemm_kernels.h"

// What bounds it: fp32 matrix instructions run on the vector ALU's multipliers (a dependent chain of them reaches 134-145 of
// 157 TFLOP/s with one to three waves per SIMD, and every vector instruction beside them is matrix time lost: four selects per
// 128 matrix cycles cost a tenth of the kernel).  So the main loop has none: operand tiles go global -> LDS by DMA with the
// base in scalar registers, LDS addresses are computed once and the stage is in the instructions' offsets (the loop is unrolled
// over the stages of 32-wide k-tiles), and a k-tile of 1024 matrix cycles has one barrier.  The values of a part of a
// k-tile are fetched under the matrix instructions of the part before it.  What the epilogue reads is fetched before the main
// loop (16 values per lane: one round trip instead of sixteen behind the stores).
// LDS formats, per operand and stage:
//   K-contiguous memory: [rows][32 k], 128 B a row = 8 chunks of 16 B, chunk c of row r at c ^ ((r >> 1) & 7).
//   k-major memory: [32 k][rows]; the 16-row blocks of a k-row change places by k % 4 (64 rows) or k / 2 % 2 (32).
// A 16x16x4 instruction's operand is sixteen rows and four k: one chunk of each row, all 64 banks once.  The same tiles on 32x32x2,
// whose operand is two of the four words of 32 rows' chunks -- every bank in use twice, half the banks not at all --, and on
// 16x16x4, four independent accumulators a wave (us): NT 2048x3072x768 92.1 / 82.8, 4096x4096x4096 1094 / 998, 2048x768x3072 (64x32
// tiles) 92.2 / 87.2; NN, one operand k-major, 82.5 / 78.8, 1013 / 964, 85.4 / 84.0; TN 4096x4096x4096 1020 / 982, short ones equal.
// (2048 tokens x 768, forward and backward of two layers: 19.05 / 18.4 ms.)
// Every element adds up its contraction one by one, k ascending, whichever instruction does it; groups and waves each add up their share of it (the
// even, resp. odd 16-wide k-tiles; one 32-wide slice) and the shares' sums are added in order.  Which kernel runs a
// problem is a matter of its shape and layout alone.
// (volatile: pairs of reads merged into one instruction have no room for the stage's offset, i.e. cost an addition each)
typedef const volatile __attribute__((address_space(3))) float lds_f32;
// WIDE: rows of 2^22 elements and more, whose tile does not fit the 32-bit offsets: 64-bit addresses, added up per load
// QUADS: read in groups of four k (16x16x4 instructions): 32-wide rows keep columns 0..15 of k % 4 >= 2 at the place of columns 16..31
template <int ROWS, bool KM, int NW = 4, bool WIDE = false, bool QUADS = false> struct F32Operand {
    using Offset = std::conditional_t<WIDE, int64_t, unsigned>;
    static constexpr int BYTES = ROWS * 32 * 4, ROUNDS = BYTES / (1024 * NW);   // NW waves load a stage
    const float* base;          // wave-uniform: the tile's first row (K-contiguous) / column (k-major), the next k-tile
    Offset off[ROUNDS];         // the lane's 16 bytes from there
    int k_lane[ROUNDS];         // ... and their k inside a k-tile
    int64_t step;
    __device__ __forceinline__ void init(const float* p, int64_t ld, int row0, int rows, int lane, int wave) {
        base = p + (KM ? row0 : (int64_t)row0 * ld);
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int q = i * NW + wave;
            if constexpr (!KM) {
                const int r = q * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
                k_lane[i] = c * 4;
                off[i] = (Offset)((int64_t)min(r, rows - 1 - row0) * ld + c * 4) * (Offset)4;
            } else {
                constexpr int CPR = ROWS / 4, RPI = 64 / CPR;   // 16-byte chunks per k-row, k-rows per instruction
                const int k = q * RPI + lane / CPR, c = (lane % CPR) ^ (!QUADS ? 0 : ROWS == 64 ? 4 * (k & 3) : 4 * ((k >> 1) & 1));
                k_lane[i] = k;
                off[i] = (Offset)((int64_t)k * ld + min(c * 4, rows - 4 - row0)) * (Offset)4;
            }
        }
        step = KM ? 32 * ld : 32;
    }
    // `left`: contraction elements from the k-tile's start (< 32: the last, ragged one); lds: LDS address of the stage
    __device__ __forceinline__ void issue(unsigned lds, int wave, int left, int lane) {
        if (!WIDE && left >= 32) {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i)
                if constexpr (!WIDE) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds + (i * NW + wave) * 1024), "v"(off[i]), "s"(base) : "m0");
        } else {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i)
                dma16_at(k_lane[i] < left ? (const unsigned char*)base + off[i] : bb_zero_line + (lane & 7) * 16, lds + (i * NW + wave) * 1024);
        }
        base += step;
    }
};
// The operand values of a wave's 32 rows: lane = row (lane & 15) of either half, k (lane >> 4) of each chunk of four.  NC: chunks of a
// k-tile the wave takes, from chunk c0 on.
template <int ROWS, bool KM, int NC> struct F32QuadReader {
    unsigned at[KM ? 2 : NC];   // LDS addresses inside stage 0; k-major: of either half
    __device__ __forceinline__ void init(unsigned lds, int row0, int c0, int lane) {
        const int r = row0 + (lane & 15), kq = lane >> 4;
        if constexpr (KM) {
#pragma unroll
            for (int i = 0; i < 2; ++i) at[i] = lds + ((4 * c0 + kq) * ROWS + ((r + 16 * i) ^ (ROWS == 64 ? 16 * kq : 16 * (kq >> 1)))) * 4;
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) at[c] = lds + r * 128 + (((c0 + c) ^ ((r >> 1) & 7)) << 4) + 4 * kq;
        }
    }
    // chunks FIRST .. FIRST + N - 1 of the stage STAGE_OFF bytes behind stage 0
    template <int STAGE_OFF, int FIRST, int N> __device__ __forceinline__ void load(float (&v)[N][2]) const {
#pragma unroll
        for (int c = 0; c < N; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                v[c][i] = KM ? *((lds_f32*)at[KM ? i : 0] + STAGE_OFF / 4 + (FIRST + c) * 4 * ROWS) : *((lds_f32*)at[KM ? 0 : FIRST + c] + STAGE_OFF / 4 + i * 16 * 32);
    }
};

// The same for 32x32x2 instructions, of a tile of 32 rows: lane = row (lane & 31), its half's k of the pairs (4 c, 4 c + 1) and
// (4 c + 2, 4 c + 3) of chunk c.
template <bool KM, int NC> struct F32Reader {
    unsigned at[KM ? 1 : NC];   // LDS addresses inside stage 0
    __device__ __forceinline__ void init(unsigned lds, int lane) {
        const int r = lane & 31, h = lane >> 5;
        if constexpr (KM) at[0] = lds + (h * 32 + r) * 4;
        else {
#pragma unroll
            for (int c = 0; c < NC; ++c) at[c] = lds + r * 128 + ((c ^ ((r >> 1) & 7)) << 4) + 4 * h;
        }
    }
    // chunks FIRST .. FIRST + N - 1 of the stage STAGE_OFF bytes behind stage 0
    template <int STAGE_OFF, int FIRST, int N> __device__ __forceinline__ void load(float (&v)[N][2]) const {
#pragma unroll
        for (int c = 0; c < N; ++c) {
            lds_f32* p = KM ? (lds_f32*)at[0] + STAGE_OFF / 4 + (FIRST + c) * 128 : (lds_f32*)at[FIRST + c] + STAGE_OFF / 4;
            v[c][0] = p[0];
            v[c][1] = p[KM ? 64 : 2];
        }
    }
};

// two stages of a 64x64 tile (32 KB), three of a 64x32 tile (36 KB): four blocks per CU either way, as the registers allow
constexpr int f32_stages(int bn) { return bn == 64 ? 2 : 3; }
constexpr int f32_gemm_lds(int bn) { return f32_stages(bn) * (64 + bn) * 128; }

// The epilogue of a lane's NR elements -- sixteen, or four of a tile that several waves finish -- (one column; register r: row m
// + STEP (r / 4) + r % 4).  `pre`: what it reads beside the product -- the operand of the epilogue kind, else the C it accumulates
// into -- fetched before the main loop; `rest`: a problem that reads both, or a masked residual, fetches the second here.  One
// branch over the kind around them, not inside: the code stays small.
template <int NR, int STEP = 8, typename V>
__device__ __forceinline__ void epilogue_f32(const GemmArgs& g, int64_t coff, int m0, int n, float bias, const float (&pre)[NR], V& v) {
    const auto row = [&](int r) { return m0 + STEP * (r >> 2) + (r & 3); };
    const bool has_opnd = epilogue_operand(g) != nullptr;
    float rest[NR], keep[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        rest[r] = pre[r];
        keep[r] = 1.0f;
    }
    if (has_opnd && g.accumulate) {
#pragma unroll
        for (int r = 0; r < NR; ++r) rest[r] = ((const float*)g.C)[coff + (int64_t)min(row(r), g.M - 1) * g.ldc + n];
    } else if (g.epilogue == BB_EPI_MUL_POS && g.resid) {
#pragma unroll
        for (int r = 0; r < NR; ++r) rest[r] = ((const float*)g.resid)[coff + (int64_t)min(row(r), g.M - 1) * g.ldaux + n];
    }
    if (g.drop.thresh) {
#pragma unroll
        for (int r = 0; r < NR; ++r) keep[r] = drop_factor(g, row(r), n);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) v[r] = v[r] * g.alpha + bias;
    float* aux = (float*)g.aux_out + coff + n;
    if (g.epilogue == BB_EPI_ACT) {
        if (g.aux_out) {
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (row(r) < g.M) aux[(int64_t)row(r) * g.ldaux] = v[r];
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] = act_f(v[r], g.act) * keep[r];
    } else if (g.epilogue == BB_EPI_ACT_DACT) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            float a, d;
            act_dact_f(v[r], g.act, a, d);
            if (row(r) < g.M) aux[(int64_t)row(r) * g.ldaux] = d * keep[r];
            v[r] = a * keep[r];
        }
    } else if (g.epilogue == BB_EPI_DACT) {
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] *= dact_f(pre[r], g.act);
    } else if (g.epilogue == BB_EPI_RESIDUAL) {
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] = v[r] * keep[r] + pre[r];
    } else if (g.epilogue == BB_EPI_MUL) {
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] *= pre[r];
    } else if (g.epilogue == BB_EPI_MUL_POS) {
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] = pre[r] > 0.f ? (g.resid ? v[r] + rest[r] : v[r]) : 0.f;
    } else {
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] *= keep[r];
    }
    float* c = (float*)g.C + coff + n;
#pragma unroll
    for (int r = 0; r < NR; ++r)
        if (row(r) < g.M) c[(int64_t)row(r) * g.ldc] = g.accumulate ? rest[r] + v[r] : v[r];
}

// (block_id: the block's index among the problem's tiles; logical_id: it is not a hardware block id, so the tile order takes it
// as it is instead of undoing the round-robin over the XCDs)
template <bool TA, bool TB, int BN, bool WIDE = false>
__device__ __forceinline__ void gemm_f32_body(const GemmArgs& g, const int block_id, const int batch_id, const bool logical_id) {
    static_assert(BN == 64 || BN == 32, "tiles: 64x64, 64x32 with the contraction shared by two groups");
    constexpr int KG = 64 / BN;
    using OpA = F32Operand<64, TA, 4, WIDE, true>;
    using OpB = F32Operand<BN, TB, 4, WIDE, true>;
    constexpr int STAGES = f32_stages(BN), STAGE = OpA::BYTES + OpB::BYTES, LOADS = OpA::ROUNDS + OpB::ROUNDS;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = KG == 1 ? wave >> 1 : 0, grp = KG == 1 ? 0 : wave >> 1;
    int tile_m, tile_n;
    if (logical_id) panel_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    else tile_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * 64, n0 = tile_n * BN;
    const int b1 = batch_id / g.nb2, b2 = batch_id % g.nb2;
    const int64_t coff = b1 * g.sC1 + b2 * g.sC2;
    OpA opa;
    OpB opb;
    opa.init((const float*)g.A + b1 * g.sA1 + b2 * g.sA2, g.lda, m0, g.M, lane, wave);
    opb.init((const float*)g.B + b1 * g.sB1 + b2 * g.sB2, g.ldb, n0, g.N, lane, wave);

    constexpr int NC = 8 / KG;   // chunks of four k of a k-tile that this wave multiplies
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t*)smem;
    F32QuadReader<64, TA, NC> ra;
    F32QuadReader<BN, TB, NC> rb;
    ra.init(lds0, wm * 32, grp * NC, lane);
    rb.init(lds0 + OpA::BYTES, wn * 32, grp * NC, lane);

    // what the epilogue reads: lane = column n + 16 j, register r = row acc_m + 16 (r / 4) + r % 4
    const int n = n0 + wn * 32 + (lane & 15), acc_m = m0 + wm * 32 + 4 * (lane >> 4);
    const float* opnd = (const float*)epilogue_operand(g);
    const int64_t ld_pre = opnd ? g.ldaux : g.ldc;
    if (!opnd && g.accumulate) opnd = (const float*)g.C;
    float bias[2] = {0.f, 0.f}, pre[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 8; ++r) pre[j][r] = 0.f;
    if (grp == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int nc = min(n + 16 * j, g.N - 1);    // clamped: what is read for a row or column past the end is not used
            if (g.bias) bias[j] = ((const float*)g.bias)[nc];
            if (opnd) {
#pragma unroll
                for (int r = 0; r < 8; ++r) pre[j][r] = opnd[coff + (int64_t)min(acc_m + 16 * (r >> 2) + (r & 3), g.M - 1) * ld_pre + nc];
            }
        }
    }

    f32x4 acc[2][2];   // [row half][column half]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int KT = (g.K + 31) / 32;
    int issued = 0, into = 0;
    auto issue = [&]() {
        const int left = g.K - issued * 32;
        opa.issue(lds0 + into, wave, left, lane);
        opb.issue(lds0 + into + OpA::BYTES, wave, left, lane);
        into = into == (STAGES - 1) * STAGE ? 0 : into + STAGE;
        ++issued;
    };
    // a k-tile is multiplied in two parts; the values of the next part -- behind the barrier that makes the next k-tile visible,
    // where it begins one -- are fetched under the matrix instructions of this one, into the other register set
    float fa[2][NC / 2][2], fb[2][NC / 2][2];
    auto multiply = [&](const float (&x)[NC / 2][2], const float (&y)[NC / 2][2]) {
#pragma unroll
        for (int c = 0; c < NC / 2; ++c)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t >> 1][t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[c][t >> 1], y[c][t & 1], acc[t >> 1][t & 1], 0, 0, 0);
    };
    // the k-tile after kt - 1 has landed (in-order completion; with three stages one more may be in flight) and every wave has
    // read that one: its stage takes the next
    auto next_tile = [&](int kt) {
        asm volatile("" ::: "memory");
        if (STAGES == 3 && kt + 1 < KT) wait_vmcnt_lgkm0<LOADS>();
        else wait_vmcnt_lgkm0<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (issued < KT) issue();
    };
    auto k_tile = [&](int kt, auto stage_c) {
        constexpr int S = decltype(stage_c)::value, NX = (S + 1) % STAGES;
        ra.template load<S * STAGE, NC / 2>(fa[1]);
        rb.template load<S * STAGE, NC / 2>(fb[1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[0], fb[0]);
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < KT) next_tile(kt + 1);
        // (behind the last k-tile: of a stage that is there, for nobody; no branch around the reads)
        ra.template load<NX * STAGE, 0>(fa[0]);
        rb.template load<NX * STAGE, 0>(fb[0]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[1], fb[1]);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (KT > 0) {
        issue();
        if (KT > 1) issue();
        if (STAGES == 3 && KT > 2) issue();
        // in-order completion: the first k-tile has landed
        asm volatile("" ::: "memory");
        if (KT > 2 && STAGES == 3) wait_vmcnt_lgkm0<2 * LOADS>();
        else if (KT > 1) wait_vmcnt_lgkm0<LOADS>();
        else wait_vmcnt_lgkm0<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        ra.template load<0, 0>(fa[0]);
        rb.template load<0, 0>(fb[0]);
        int kt = 0;
        for (; kt + STAGES <= KT; kt += STAGES) {
            k_tile(kt, std::integral_constant<int, 0>{});
            k_tile(kt + 1, std::integral_constant<int, 1>{});
            if constexpr (STAGES == 3) k_tile(kt + 2, std::integral_constant<int, 2>{});
        }
        if (kt < KT) k_tile(kt, std::integral_constant<int, 0>{});
        if (STAGES == 3 && kt + 1 < KT) k_tile(kt + 1, std::integral_constant<int, 1>{});
    }
    if constexpr (KG > 1) {
        // group 1's partial tile through the (drained) stages
        f32x4* part = (f32x4*)smem + wm * (4 * 64);
        __syncthreads();
        if (grp == 1) {
#pragma unroll
            for (int t = 0; t < 4; ++t) part[t * 64 + lane] = acc[t >> 1][t & 1];
        }
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 other = part[t * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t >> 1][t & 1][e] += other[e];
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = acc[r >> 2][j][r & 3];
        if (n + 16 * j < g.N) epilogue_f32<8, 16>(g, coff, acc_m, n + 16 * j, bias[j], pre[j], v);
    }
}

template <bool TA, bool TB, int BN, bool WIDE = false>
__global__ __launch_bounds__(256, WIDE ? 2 : 4) void gemm_f32_kernel(const GemmArgs g) {
    gemm_f32_body<TA, TB, BN, WIDE>(g, blockIdx.x, blockIdx.z, false);
}
// several unbatched problems in one launch (the weight gradients of an fp32 layer)
template <bool TA, bool TB>
__global__ __launch_bounds__(256, 4) void gemm_f32_grouped_kernel(const GroupedArgs G) {
    const int lid = grouped_place<4>(G);
    if (lid < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && lid >= G.first_block[pi + 1]) ++pi;
    gemm_f32_body<TA, TB, 64>(G.p[pi], lid - G.first_block[pi], 0, true);
}

// Problems of few tiles and a contraction of at most 128: 32x32 tiles, each of the four waves of a block one 32-wide slice.
// What bounds such a problem is a chain -- per k-tile a wait for the loads, a barrier and 1024 cycles of dependent matrix
// instructions, on a handful of CUs.  Here everything is in flight at once, nobody waits for anybody, and the chain is one
// slice long on four times the CUs; the four partial tiles meet in LDS, are added in wave order, and each wave finishes eight
// rows.  (us against the 64x64 tiles: see pick_f32_wave; the error against 64 bits at K = 128: 2.0e-7 -> 1.1e-7.)
constexpr int kF32Waves = 4, kF32WaveK = kF32Waves * 32;
constexpr int kF32WaveLds = kF32Waves * 2 * 32 * 128;
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_f32_wave_body(const GemmArgs& g, const int block_id, const int batch_id, const bool logical_id) {
    using OpA = F32Operand<32, TA, 1>;
    using OpB = F32Operand<32, TB, 1>;
    constexpr int KW = kF32Waves, SLICE = OpA::BYTES + OpB::BYTES;
    static_assert(KW * SLICE == kF32WaveLds && SLICE >= 32 * 32 * 4, "a wave's partial tile takes the place of its slice");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tile_m, tile_n;
    if (logical_id) panel_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    else tile_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * 32, n0 = tile_n * 32;
    const int b1 = batch_id / g.nb2, b2 = batch_id % g.nb2;
    const int64_t coff = b1 * g.sC1 + b2 * g.sC2;
    OpA opa;
    OpB opb;
    opa.init((const float*)g.A + b1 * g.sA1 + b2 * g.sA2, g.lda, m0, g.M, lane, 0);
    opb.init((const float*)g.B + b1 * g.sB1 + b2 * g.sB2, g.ldb, n0, g.N, lane, 0);
    opa.base += wave * opa.step;
    opb.base += wave * opb.step;
    const unsigned lds = (unsigned)(uintptr_t)(lds_ptr_t*)smem + wave * SLICE;
    F32Reader<TA, 8> ra;
    F32Reader<TB, 8> rb;
    ra.init(lds, lane);
    rb.init(lds + OpA::BYTES, lane);
    const int left = g.K - wave * 32;
    if (left > 0) {
        opa.issue(lds, 0, left, lane);
        opb.issue(lds + OpA::BYTES, 0, left, lane);
    }

    // what the epilogue reads, for the rows this wave will finish: register e = row acc_m + e
    const int n = n0 + (lane & 31), acc_m = m0 + 8 * wave + 4 * (lane >> 5), nc = min(n, g.N - 1);
    const float* opnd = (const float*)epilogue_operand(g);
    const int64_t ld_pre = opnd ? g.ldaux : g.ldc;
    if (!opnd && g.accumulate) opnd = (const float*)g.C;
    const float bias = g.bias ? ((const float*)g.bias)[nc] : 0.f;
    float pre[4] = {0.f, 0.f, 0.f, 0.f};
    if (opnd) {
#pragma unroll
        for (int e = 0; e < 4; ++e) pre[e] = opnd[coff + (int64_t)min(acc_m + e, g.M - 1) * ld_pre + nc];
    }

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (left > 0) {
        asm volatile("" ::: "memory");
        wait_vmcnt_lgkm0<0>();
        asm volatile("" ::: "memory");
        float x[8][2], y[8][2];
        ra.template load<0, 0>(x);
        rb.template load<0, 0>(y);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[c][i], y[c][i], acc, 0, 0, 0);
    }

    float* part = (float*)smem;
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave * (SLICE / 4) + r * 64 + lane] = acc[r];
    __syncthreads();
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = part[(4 * wave + e) * 64 + lane];
#pragma unroll
        for (int p = 1; p < KW; ++p) v[e] += part[p * (SLICE / 4) + (4 * wave + e) * 64 + lane];
    }
    if (n < g.N) epilogue_f32<4>(g, coff, acc_m, n, bias, pre, v);
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256, 4) void gemm_f32_wave_kernel(const GemmArgs g) {
    gemm_f32_wave_body<TA, TB>(g, blockIdx.x, blockIdx.z, false);
}
template <bool TA, bool TB>
__global__ __launch_bounds__(256, 4) void gemm_f32_wave_grouped_kernel(const GroupedArgs G) {
    const int lid = grouped_place<4>(G);
    if (lid < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && lid >= G.first_block[pi + 1]) ++pi;
    gemm_f32_wave_body<TA, TB>(G.p[pi], lid - G.first_block[pi], 0, true);
}

// Problems of few 64x64 tiles: each tile as four blocks of 32x32, a wave 16x16 of it by v_mfma_f32_16x16x4_f32.  What bounds such
// a problem is the chain of one tile: a 64x64 tile's wave spends 32 matrix cycles on every k, this one 8 on four times the CUs,
// and four k-tiles of 64 are in flight from the start (us against the larger tiles: see pick_f32_quarter).  Both instructions add
// their k one by one, ascending (checked bit for bit against a chain of multiply-adds), so the result has the bits of the larger
// tile: which kernel runs a product changes none of them.
// KG: groups of four waves that share the contraction as those of the 64x32 tiles do (16-wide halves of every 32, added in order).
constexpr int kF32QuarterStages = 4;
constexpr int kF32QuarterLds = kF32QuarterStages * 2 * 2 * 32 * 128;
template <bool TA, bool TB, int KG>
__device__ __forceinline__ void gemm_f32_quarter_body(const GemmArgs& g, const int block_id, const int batch_id, const bool logical_id) {
    constexpr int NW = 4 * KG, NST = kF32QuarterStages;
    using OpA = F32Operand<32, TA, 4, false, true>;     // a k-tile of 32: four instructions
    using OpB = F32Operand<32, TB, 4, false, true>;
    constexpr int TILE = OpA::BYTES + OpB::BYTES, STAGE = 2 * TILE, LOADS = 16 / NW;   // instructions a wave and stage
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int quad = wave & 3, grp = wave >> 2, wm = quad & 1, wn = quad >> 1;
    int tile_m, tile_n;
    if (logical_id) panel_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    else tile_coords(block_id, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * 32, n0 = tile_n * 32;
    const int b1 = batch_id / g.nb2, b2 = batch_id % g.nb2;
    const int64_t coff = b1 * g.sC1 + b2 * g.sC2;
    // a stage is two 32-wide k-tiles of both operands; with one group every wave loads a quarter of each, with two a group loads one k-tile
    OpA opa;
    OpB opb;
    opa.init((const float*)g.A + b1 * g.sA1 + b2 * g.sA2, g.lda, m0, g.M, lane, quad);
    opb.init((const float*)g.B + b1 * g.sB1 + b2 * g.sB2, g.ldb, n0, g.N, lane, quad);
    if (KG == 2 && grp == 1) {
        opa.base += opa.step;
        opb.base += opb.step;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t*)smem;

    // what the epilogue reads: lane = column, register r = row acc_m + r
    const int n = n0 + wn * 16 + (lane & 15), acc_m = m0 + wm * 16 + 4 * (lane >> 4), nc = min(n, g.N - 1);
    const float* opnd = (const float*)epilogue_operand(g);
    const int64_t ld_pre = opnd ? g.ldaux : g.ldc;
    if (!opnd && g.accumulate) opnd = (const float*)g.C;
    float bias = 0.f, pre[4] = {0.f, 0.f, 0.f, 0.f};
    if (grp == 0) {
        if (g.bias) bias = ((const float*)g.bias)[nc];
        if (opnd) {
#pragma unroll
            for (int e = 0; e < 4; ++e) pre[e] = opnd[coff + (int64_t)min(acc_m + e, g.M - 1) * ld_pre + nc];
        }
    }

    const int KS = (g.K + 63) / 64;   // stages of 64
    int into = 0, issued = 0;
    auto issue = [&]() {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (KG == 2 && h != grp) continue;
            const int left = g.K - issued * 64 - h * 32;
            const unsigned at = lds0 + into + h * TILE;
            opa.issue(at, quad, left, lane);
            opb.issue(at + OpA::BYTES, quad, left, lane);
        }
        if (KG == 2) {   // the other group's k-tile
            opa.base += opa.step;
            opb.base += opb.step;
        }
        into = into == (NST - 1) * STAGE ? 0 : into + STAGE;
        ++issued;
    };
    // stage s has landed when at most (stages issued behind it) x LOADS are in flight: completion is in order
    auto landed = [&](int behind) {
        asm volatile("" ::: "memory");
        if (behind >= 3) wait_vmcnt_lgkm0<3 * LOADS>();
        else if (behind == 2) wait_vmcnt_lgkm0<2 * LOADS>();
        else if (behind == 1) wait_vmcnt_lgkm0<LOADS>();
        else wait_vmcnt_lgkm0<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    static_assert(NST == 4, "landed()");

    constexpr int NC = 8 / KG;         // chunks of four k of a k-tile that this wave multiplies
    const int fr = lane & 15, kq = lane >> 4;
    unsigned at_a[TA ? 1 : NC], at_b[TB ? 1 : NC];
    const int ra = wm * 16 + fr, rb = wn * 16 + fr;
    if constexpr (TA) at_a[0] = lds0 + ((4 * grp * NC + kq) * 32 + (ra ^ (16 * (kq >> 1)))) * 4;
    else {
#pragma unroll
        for (int c = 0; c < NC; ++c) at_a[c] = lds0 + ra * 128 + (((grp * NC + c) ^ ((ra >> 1) & 7)) << 4) + 4 * kq;
    }
    if constexpr (TB) at_b[0] = lds0 + OpA::BYTES + ((4 * grp * NC + kq) * 32 + (rb ^ (16 * (kq >> 1)))) * 4;
    else {
#pragma unroll
        for (int c = 0; c < NC; ++c) at_b[c] = lds0 + OpA::BYTES + rb * 128 + (((grp * NC + c) ^ ((rb >> 1) & 7)) << 4) + 4 * kq;
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float fa[2][NC], fb[2][NC];
    auto load = [&](auto off_c, float (&a)[NC], float (&b)[NC]) {
        constexpr int OFF = decltype(off_c)::value;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            a[c] = TA ? *((lds_f32*)at_a[0] + OFF / 4 + c * 128) : *((lds_f32*)at_a[TA ? 0 : c] + OFF / 4);
            b[c] = TB ? *((lds_f32*)at_b[0] + OFF / 4 + c * 128) : *((lds_f32*)at_b[TB ? 0 : c] + OFF / 4);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const float (&a)[NC], const float (&b)[NC]) {
#pragma unroll
        for (int c = 0; c < NC; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c], b[c], acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // a stage: its second k-tile is read under the first one's products, the next stage's first -- behind the barrier that makes it
    // visible and frees the stage before this one -- under the second one's
    auto stage = [&](int s, auto stage_c) {
        constexpr int S = decltype(stage_c)::value, NX = (S + 1) % NST;
        load(std::integral_constant<int, S * STAGE + TILE>{}, fa[1], fb[1]);
        multiply(fa[0], fb[0]);
        if (s + 1 < KS) {
            landed(issued - s - 2);
            if (issued < KS) issue();
        }
        load(std::integral_constant<int, NX * STAGE>{}, fa[0], fb[0]);   // (behind the last stage: of one that is there, for nobody)
        multiply(fa[1], fb[1]);
    };
    if (KS > 0) {
        for (int p = 0; p < NST && p < KS; ++p) issue();
        landed(issued - 1);
        load(std::integral_constant<int, 0>{}, fa[0], fb[0]);
        int s = 0;
        for (; s + NST <= KS; s += NST) {
            stage(s, std::integral_constant<int, 0>{});
            stage(s + 1, std::integral_constant<int, 1>{});
            stage(s + 2, std::integral_constant<int, 2>{});
            stage(s + 3, std::integral_constant<int, 3>{});
        }
        if (s < KS) stage(s, std::integral_constant<int, 0>{});
        if (s + 1 < KS) stage(s + 1, std::integral_constant<int, 1>{});
        if (s + 2 < KS) stage(s + 2, std::integral_constant<int, 2>{});
    }
    if constexpr (KG > 1) {
        float* part = (float*)smem + quad * (4 * 64);
        __syncthreads();
        if (grp == 1) {
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r * 64 + lane] = acc[r];
        }
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += part[r * 64 + lane];
    }
    if (n < g.N) epilogue_f32<4>(g, coff, acc_m, n, bias, pre, acc);
}
template <bool TA, bool TB, int KG>
__global__ __launch_bounds__(256 * KG, 2) void gemm_f32_quarter_kernel(const GemmArgs g) {
    gemm_f32_quarter_body<TA, TB, KG>(g, blockIdx.x, blockIdx.z, false);
}
// weight gradients of few tiles over many rows
__global__ __launch_bounds__(256, 2) void gemm_f32_quarter_grouped_kernel(const GroupedArgs G) {
    const int lid = grouped_place<4>(G);
    if (lid < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && lid >= G.first_block[pi + 1]) ++pi;
    gemm_f32_quarter_body<true, true, 1>(G.p[pi], lid - G.first_block[pi], 0, true);
}
