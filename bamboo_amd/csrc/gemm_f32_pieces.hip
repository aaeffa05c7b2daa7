// fp32 products on v_mfma_f32_16x16x32_bf16: every operand value as the sum of three bf16 pieces.
//
// Why: fp32 matrix instructions do 157 TFLOP/s, bf16 ones 2500, and six of these make one fp32 product: x = x0 + x1 + x2 exactly
// (three times eight bits, each piece the nearest bf16 of what the ones before leave), and of the nine products of two such sums the three of
// x1 y2, x2 y1 and x2 y2 are below 2^-24 of x y and left out.  (G. Henry, P. Tang, A. Heinecke: Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations, ARITH 2019.)  x0 y0 has an accumulator of its own, the five small ones share another: the large sum is
// rounded once per instruction instead of once per k, so that the result is nearer to the exact one than that of the fp32 instructions (2-norm
// against 64 bits, K 64 / 768 / 3072 / 8192: 4.9e-8, 1.6e-7, 3.4e-7, 5.7e-7 against 1.5e-7, 3.5e-7, 7.0e-7, 1.15e-6; values of one, 20 and 40
// octaves in either operand, K 772: 1.6e-7, 1.9e-7, 1.6e-7 against 3.5e-7, 2.9e-7, 1.6e-7).  Beyond that the instruction's way of adding shows: it drops, towards
// minus infinity, what lies below the last bit of its largest addend (80 octaves: 1.3e-7 against 1.2e-7).
//
// Range: a last piece lies up to 23 bits below its value, and bf16 has nothing below 2^-133.  So values are taken times 2^16: the last bit of the
// smallest, 2^-149, is then a bf16, and every fp32 value the sum of its pieces (the instruction keeps subnormals); the sums carry 2^32, taken out of
// the result.  Without that, normal values of 2^-120 lose eleven bits (2-norm 3.5e-5).  It costs two of thirteen instructions of a pair's splitting,
// 2.5 % of a product.
//
// What leaves the range at its upper end -- values from 2^112, sums from 2^96 on, infinities, NaN -- is found in the result: it makes its row or column
// of the tile, or the one sum, not finite.  A wave that finds such a sum makes its part of the tile again, on fp32 instructions (pieces_again).
//
// What bounds it: what the waves issue -- beside every matrix instruction about two for the splitting (an instruction is free beside the first 16
// cycles' two) --, LDS' write path (64 bytes a cycle) and the waits at the barrier: counted in a stage of 768 columns, a CU in use has the matrix pipe
// 39 to 49 % and the vector ALU 42 to 51 % busy, at 2.23 to 2.34 of 2.4 GHz.  192 tiles on 256 CUs and rounds of 288 take a quarter on top.
//
// Loop: 32-wide k-tiles, global memory -> registers four k-tiles ahead, split there (a value once in a block), pieces -> LDS, two stages.  The
// splitting is spread over the matrix instructions of a whole k-tile, whichever stage it goes to; one barrier a k-tile (see step).
// LDS: three planes an operand.  k-contiguous: 64 bytes a row, its chunks of 16 swizzled by the row's block of four (no bank conflict counted);
// k-major: as in gemm_m16.h.  The product is made transposed: a lane holds four neighbouring columns of a row of C.
#include "gemm_f32_pieces.h"
#include "gemm_m16.h"

constexpr float kPiecesScale = 65536.f;     // of either operand, see above
// chunk swizzle of 64-byte rows by the row: 0, 2, 3, 1 by its block of four
__device__ __forceinline__ int pieces_row_swizzle(int r) { return ((r >> 1) & 2) ^ ((r >> 3) & 1) * 3; }
// A thread's share of one operand tile, BR rows (columns of a k-major operand) x 32 k: fours of neighbouring values, neighbouring lanes next to
// each other in memory.
template <int BR, int NT, bool KM> struct PiecesOperand {
    static constexpr int PLANE = BR * 64, BYTES = 3 * PLANE, FOURS = BR * 8 / NT, CPR = KM ? BR / 4 : 8, DOWN = NT / CPR;   // fours a row, rows between a thread's
    static_assert(BR * 8 % NT == 0 && (KM ? DOWN % 8 == 0 : DOWN % 16 == 0), "whole fours a thread, swizzled alike");
    const float* base;
    int64_t step;
    unsigned off[FOURS];      // bytes from base
    int k_at, lds0;

    __device__ __forceinline__ void init(const float* p, int64_t ld, int row0, int rows, int tid) {
        const int r = tid / CPR, c = tid % CPR;
        k_at = KM ? r : c * 4;
        if constexpr (!KM) lds0 = r * 64 + (((c >> 1) ^ pieces_row_swizzle(r)) << 4) + (c & 1) * 8;
        else lds0 = r * (BR * 2) + (((c >> 1) ^ m16_k_swizzle<BR, false>(r)) << 4) + (c & 1) * 8;
#pragma unroll
        for (int i = 0; i < FOURS; ++i)
            off[i] = KM ? ((unsigned)(r + i * DOWN) * (unsigned)ld + min(c * 4, rows - 4 - row0)) * 4 : ((unsigned)min(r + i * DOWN, rows - 1 - row0) * (unsigned)ld + c * 4) * 4;
        base = p + (KM ? row0 : (int64_t)row0 * ld);
        step = KM ? 32 * ld : 32;
    }
    template <int I> __device__ __forceinline__ int lds() const {
        constexpr int TURN = KM ? ((I * DOWN >> 3) & 1) << 5 : 0;     // (every eighth k the swizzle changes, see m16_k_swizzle)
        return (lds0 ^ TURN) + I * DOWN * (KM ? BR * 2 : 64);
    }
    // four I of the next k-tile, of which `left` k are there (<= 0: none); what lies behind them reads as zero (an offset past the descriptor's range)
    template <int I> __device__ __forceinline__ void load(float (&v)[FOURS][4], int left) {
        const auto desc = __builtin_amdgcn_make_buffer_rsrc((void*)m16_uniform((const char*)base), 0, 0x80000000u, 0x00020000);
        const unsigned o = k_at < left - (KM ? I * DOWN : 0) ? off[I] : 0x80000000u;
        const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(desc, o, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[I][e] = x[e];
        if constexpr (I == FOURS - 1) base += step;
    }
};
// a wave's fragments of one plane, T of 16 rows x 32 k, from tile row wbase on; lane l holds row l % 16, k = 8 (l / 16) .. + 7
template <int BR, int T, bool KM> struct PiecesFrags {
    M16Frags<BR, T, KM, false> km;
    int off;
    __device__ __forceinline__ void init(int wbase, int lane) {
        if constexpr (KM) km.init(wbase, lane);
        else {
            const int row = wbase + (lane & 15);
            off = row * 64 + (((lane >> 4) ^ pieces_row_swizzle(row)) << 4);
        }
    }
    __device__ __forceinline__ bf16x8 load(const unsigned char* plane, int t) const {
        if constexpr (KM) return km.load(plane, t, 0);
        else return *(const bf16x8*)(plane + off + t * 1024);
    }
};

// A wave's part of a tile on fp32 instructions, from memory.  A lane holds four k of a row of A, and of a row (BKM: column) of B: 16 k are four
// instructions; the even and the odd sixteens have a sum each, as where two groups share a contraction (gemm_f32.h).  What bounds it is the latency
// of its loads, 16 k ahead of their use; nothing is staged: sixteen lanes read 16 lines (k-major: one), and the waves of a row or column of waves
// the same ones.  The whole product, us, all values finite / one NaN in A / all NaN (before, one element's multiply-adds a lane): NT 2048x3072x768
// 66 / 108 (887) / 215 (3391), NN 2048x768x3072 78 / 183 (1985) / 251 (3594), a weight gradient 3072x768x2048 79 / 223 (3070) / 308 (4369); the
// fp32 kernels 85, 85 and 102 on any values.
template <bool KM> __device__ __forceinline__ f32x4 pieces_four(const float* p, int64_t ld, int k, int K) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!KM) {
        if (k < K) v = *(const f32x4*)(p + k);       // (whole fours: a k-contiguous operand has K % 4 == 0)
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k + e < K) v[e] = p[(int64_t)(k + e) * ld];
    }
    return v;
}
template <int TM, int TN, bool AKM, bool BKM> __device__ __forceinline__ void pieces_again(const GemmArgs& g, int row0, int col0, int lane, f32x4 (&acc)[TM][TN], f32x4 (&odd)[TM][TN]) {
    const float *A[TM], *B[TN];
    f32x4 a[2][TM], b[2][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = min(row0 + i * 16 + (lane & 15), g.M - 1);
        A[i] = (const float*)g.A + (AKM ? m : (int64_t)m * g.lda);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = min(col0 + j * 16 + (lane & 15), g.N - 1);
        B[j] = (const float*)g.B + (BKM ? n : (int64_t)n * g.ldb);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = odd[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int s, int k) {
#pragma unroll
        for (int i = 0; i < TM; ++i) a[s][i] = pieces_four<AKM>(A[i], g.lda, k, g.K);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[s][j] = pieces_four<BKM>(B[j], g.ldb, k, g.K);
    };
    auto add = [&](int s, f32x4 (&to)[TM][TN]) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[s][j][e], a[s][i][e], to[i][j], 0, 0, 0);
    };
    int k = 4 * (lane >> 4);
    fetch(0, k);
    for (int left = g.K; left > 0; left -= 32, k += 32) {
        fetch(1, k + 16);
        add(0, acc);
        fetch(0, k + 32);
        add(1, odd);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += odd[i][j];
}

// four neighbouring elements of a row of C; the epilogue of epilogue_f32
__device__ __forceinline__ void pieces_epilogue(const GemmArgs& g, int m, int n, f32x4 v) {
    const int64_t ci = (int64_t)m * g.ldc + n, xi = (int64_t)m * g.ldaux + n;
    float keep[4] = {1.f, 1.f, 1.f, 1.f};
    if (g.drop.thresh) {
#pragma unroll
        for (int e = 0; e < 4; ++e) keep[e] = drop_factor(g, m, n + e);
    }
    const f32x4 bias = g.bias ? *(const f32x4*)((const float*)g.bias + n) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] * g.alpha + bias[e];
    const float* opnd = (const float*)epilogue_operand(g);
    const f32x4 x = opnd ? *(const f32x4*)(opnd + xi) : f32x4{0.f, 0.f, 0.f, 0.f};
    if (g.epilogue == BB_EPI_ACT) {
        if (g.aux_out) *(f32x4*)((float*)g.aux_out + xi) = v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = act_f(v[e], g.act) * keep[e];
    } else if (g.epilogue == BB_EPI_ACT_DACT) {
        f32x4 d4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float a, d;
            act_dact_f(v[e], g.act, a, d);
            d4[e] = d * keep[e];
            v[e] = a * keep[e];
        }
        *(f32x4*)((float*)g.aux_out + xi) = d4;
    } else if (g.epilogue == BB_EPI_DACT) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= dact_f(x[e], g.act);
    } else if (g.epilogue == BB_EPI_RESIDUAL) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * keep[e] + x[e];
    } else if (g.epilogue == BB_EPI_MUL) {
        v *= x;
    } else if (g.epilogue == BB_EPI_MUL_POS) {
        if (g.resid) v += *(const f32x4*)((const float*)g.resid + xi);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[e] > 0.f ? v[e] : 0.f;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= keep[e];
    }
    f32x4* c = (f32x4*)((float*)g.C + ci);
    *c = g.accumulate ? *c + v : v;
}

template <int TM, int TN, int WM, int WN, bool AKM, bool BKM>
__device__ __forceinline__ void gemm_f32_pieces_body(const GemmArgs& g, const int block_id, const bool logical_id) {
    constexpr int NT = WM * WN * 64, BM = WM * TM * 16, BN = WN * TN * 16;
    using OpA = PiecesOperand<BM, NT, AKM>;
    using OpB = PiecesOperand<BN, NT, BKM>;
    constexpr int STAGE = OpA::BYTES + OpB::BYTES, PARTS = (OpA::FOURS + OpB::FOURS) * 16, NM = TM * TN * 6, AHEAD = 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    if (logical_id) panel_coords<8>(block_id, g.tiles_m, g.tiles_n, tm, tn);
    else tile_coords<8>(block_id, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    OpA opa;
    OpB opb;
    opa.init((const float*)g.A, g.lda, m0, g.M, tid);
    opb.init((const float*)g.B, g.ldb, n0, g.N, tid);
    PiecesFrags<BM, TM, AKM> fa;
    PiecesFrags<BN, TN, BKM> fb;
    fa.init(wave / WN * (TM * 16), lane);
    fb.init(wave % WN * (TN * 16), lane);

    f32x4 large[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) large[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    struct Held {
        float a[OpA::FOURS][4], b[OpB::FOURS][4];
    } held[AHEAD];
    int left = g.K;       // k from the next k-tile to be loaded on
    constexpr int LOADS = OpA::FOURS + OpB::FOURS;
    auto load = [&](auto i_c, Held& h) {
        constexpr int I = decltype(i_c)::value;
        if constexpr (I < OpA::FOURS) opa.template load<I>(h.a, left);
        else opb.template load<I - OpA::FOURS>(h.b, left);
        if constexpr (I == LOADS - 1) left -= 32;
    };
    auto load_all = [&](Held& h) { static_for([&](auto i) { load(i, h); }, std::make_integer_sequence<int, LOADS>{}); };
    // The pieces of a pair of values are made in eight parts of one or two instructions (times kPiecesScale; nearest bf16; the same as fp32; what they
    // leave; again; the upper halves of what those leave), two pairs in turn; a plane's pieces of a four go into the stage when it is whole.  A k-tile's parts are
    // spread evenly over NM slots, a matrix instruction each: two vector instructions beside one cost it nothing, more four cycles each.
    // (v_dot2_f32_bf16 would make two parts one, but waits for the matrix pipe: 17 cycles.)
    typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
    u32x2 made[3];
    float near[2][2];
    auto part = [&](auto n_c, Held& h, unsigned char* st) {
        constexpr int N = decltype(n_c)::value, Q = N / 16 * 2 + N % 2, at = N % 16 / 2 - 1, p = at / 3, c = Q / 2, q = Q % 2, e = q * 2;
        constexpr bool OF_A = c < OpA::FOURS;
        auto& v = [&]() -> auto& {
            if constexpr (OF_A) return h.a[c];
            else return h.b[c - OpA::FOURS];
        }();
        if constexpr (at < 0) {
            v[e] *= kPiecesScale;
            v[e + 1] *= kPiecesScale;
        } else if constexpr (at % 3 == 1) {
            near[Q % 2][0] = __uint_as_float(made[p][q] << 16);
            near[Q % 2][1] = __uint_as_float(made[p][q] & 0xffff0000u);
        } else if constexpr (at % 3 == 2) {
            v[e] -= near[Q % 2][0];
            v[e + 1] -= near[Q % 2][1];
        } else {
            made[p][q] = p == 2 ? __builtin_amdgcn_perm(__float_as_uint(v[e + 1]), __float_as_uint(v[e]), 0x07060302) : pack2bf(v[e], v[e + 1]);
            if constexpr (q == 1) {
                if constexpr (OF_A) *(u32x2*)(st + p * OpA::PLANE + opa.template lds<c>()) = made[p];
                else *(u32x2*)(st + OpA::BYTES + p * OpB::PLANE + opb.template lds<c - OpA::FOURS>()) = made[p];
            }
        }
    };
    auto split = [&](auto slot_c, Held& h, unsigned char* st) {
        constexpr int SLOT = decltype(slot_c)::value, FIRST = PARTS * SLOT / NM;
        static_for([&](auto d) { part(std::integral_constant<int, FIRST + decltype(d)::value>{}, h, st); }, std::make_integer_sequence<int, PARTS * (SLOT + 1) / NM - FIRST>{});
    };
    auto meet = [&]() {      // what this wave wrote to LDS is there, and what it read has come; then everybody's
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    bf16x8 fra[2][3], frb[2][TN][3];
    auto read_a = [&](const unsigned char* st, int i) {
#pragma unroll
        for (int p = 0; p < 3; ++p) fra[i & 1][p] = fa.load(st + p * OpA::PLANE, i);
    };
    // k-tile t, multiplied from stage t % 2.  The barrier stands behind the last read of that stage: in front of it the last values of k-tile t + 1
    // go into the other one, behind it the first values of k-tile t + 2 into this one, the first fragments of k-tile t + 1 are read, and the registers
    // that held k-tile t + 1 are loaded again.
    constexpr int BARRIER = TM > 2 ? NM * 3 / 4 : NM * 5 / 8, LAST = NM - 6 * TN, FIRST_B = LAST > BARRIER ? BARRIER : BARRIER + 1;
    static_assert(FIRST_B + 3 * TN <= NM && BARRIER > 6 * TN * (TM - 2), "reads in front of and behind the barrier");
    auto step = [&](auto t_c) {
        constexpr int T = decltype(t_c)::value, S = T % 2;
        const unsigned char* cur = smem + S * STAGE;
        unsigned char* nxt = smem + (1 - S) * STAGE;
        static_for(
            [&](auto m_c) {
                constexpr int m = decltype(m_c)::value, i = m / (6 * TN), w = m / TN % 6, j = m % TN;
                if constexpr (m == BARRIER) meet();
                if constexpr (m % (6 * TN) == 0 && i + 1 < TM) read_a(cur, i + 1);
                if constexpr (m == (LAST > BARRIER ? LAST : BARRIER)) read_a(nxt, 0);
                if constexpr (m >= FIRST_B && m < FIRST_B + 3 * TN) frb[1 - S][(m - FIRST_B) % TN][(m - FIRST_B) / TN] = fb.load(nxt + OpA::BYTES + (m - FIRST_B) / TN * OpB::PLANE, (m - FIRST_B) % TN);
                constexpr int pa[6] = {0, 0, 2, 1, 0, 1}, pb[6] = {0, 2, 0, 1, 1, 0};
                f32x4& acc = w == 0 ? large[i][j] : small[i][j];
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frb[S][j][pb[w]], fra[i & 1][pa[w]], acc, 0, 0, 0);
                if constexpr (m < BARRIER) split(std::integral_constant<int, NM - BARRIER + m>{}, held[(T + 1) % AHEAD], nxt);
                else split(std::integral_constant<int, m - BARRIER>{}, held[(T + 2) % AHEAD], smem + S * STAGE);
                if constexpr (m >= BARRIER)
                    static_for([&](auto d) { load(std::integral_constant<int, LOADS * (m - BARRIER) / (NM - BARRIER) + decltype(d)::value>{}, held[(T + 1) % AHEAD]); },
                               std::make_integer_sequence<int, LOADS * (m - BARRIER + 1) / (NM - BARRIER) - LOADS * (m - BARRIER) / (NM - BARRIER)>{});
                __builtin_amdgcn_sched_barrier(0);
            },
            std::make_integer_sequence<int, NM>{});
    };

    const int KT = (g.K + 31) / 32;
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) load_all(held[t]);
    static_for([&](auto s) { split(s, held[0], smem); }, std::make_integer_sequence<int, NM>{});
    meet();
    load_all(held[0]);
    read_a(smem, 0);
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j) frb[0][j][p] = fb.load(smem + OpA::BYTES + p * OpB::PLANE, j);
    static_for([&](auto s) { split(s, held[1], smem + STAGE); }, std::make_integer_sequence<int, NM - BARRIER>{});
    static_assert(AHEAD == 2 || AHEAD == 4, "the loop below");
    for (int kt = 0;;) {
        step(std::integral_constant<int, 0>{});
        if (++kt >= KT) break;
        step(std::integral_constant<int, 1>{});
        if (++kt >= KT) break;
        if constexpr (AHEAD == 4) {
            step(std::integral_constant<int, 2>{});
            if (++kt >= KT) break;
            step(std::integral_constant<int, 3>{});
            if (++kt >= KT) break;
        }
    }

    const int row = m0 + wave / WN * (TM * 16) + (lane & 15), col = n0 + wave % WN * (TN * 16) + 4 * (lane >> 4);
    bool finite = true;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            large[i][j] += small[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) finite = finite && fabsf(large[i][j][e]) < __builtin_inff();
        }
    const bool again = __any(!finite);
    const float unscale = again ? 1.f : 1.f / (kPiecesScale * kPiecesScale);
    if (again) pieces_again<TM, TN, AKM, BKM>(g, m0 + wave / WN * (TM * 16), n0 + wave % WN * (TN * 16), lane, large, small);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = row + i * 16;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = col + j * 16;
            if (m >= g.M || n >= g.N) continue;
            pieces_epilogue(g, m, n, large[i][j] * unscale);
        }
    }
}
template <int TM, int TN, int WM, int WN, bool AKM, bool BKM>
__global__ __launch_bounds__(WM* WN * 64) void gemm_f32_pieces_kernel(const GemmArgs g) {
    gemm_f32_pieces_body<TM, TN, WM, WN, AKM, BKM>(g, blockIdx.x, false);
}
// a layer's weight gradients in one launch
template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(WM* WN * 64) void gemm_f32_pieces_grouped_kernel(const GroupedArgs G) {
    const int id = grouped_place<WM * WN>(G);
    if (id < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && id >= G.first_block[pi + 1]) ++pi;
    gemm_f32_pieces_body<TM, TN, WM, WN, true, true>(G.p[pi], id - G.first_block[pi], true);
}

// All of a launch's problems, or one of any layout.  By an estimate of both ways, operands and outputs not in the caches.  Pieces: rounds (one tile a
// CU) of K steps, and K steps by the share of the CUs that have a tile.  fp32 instructions: K steps of the fullest CU by how many 64x64 (64x32,
// pick_f32_split) tiles it has, four of which run at a time, one alone at two thirds of their rate.  Fitted to 2900 products (100..8000 rows, 64..6400
// columns, K 32..4096) and the weight gradients of 3500 layers and 900 single ones; the estimates are off by 10, 5 and 4 % (2-norm), which is what the
// lines (a launch of few k-tiles is its epilogue: 5 %) allow for.  Where both tiles come out alike it is 128x128: 128x64 split A's values twice as often, which
// other work on the CUs feels (a stage of 2048x2304x768 and 2048x3072x768 products, two streams: 15.5 and 16.9 ms).  Of the products two in
// a thousand are more than 3 % slower on pieces than on fp32 instructions, at most 12 %, of the weight gradients none more than 5 %; the line before, by
// flops, had 45 and 75 in a thousand, up to 27 and 30 %.
// us, fp32 / 128x128 / 128x64 (the one taken marked; - what the line before took and this does not):
//     NT 2048x3072x768 88 / 63* / 65   2048x768x768 25 / 30 / 21*   2048x768x3072 84 / 99 / 70*   2048x1024x256 14.1 / 14.5 / 11.0*
//        2048x256x1024 16* / 36 / 26   512x512x512 8* / 21 / 15      4096x4096x4096 990 / 630* / 800   2048x2304x768 75.3 / 69.0* / 67.8
//     NN 2048x3072x768 78 / 63* / 66   2048x768x3072 82 / 101 / 73*  2048x768x2304 62 / 77 / 56*   1305x1536x384 20.0* / 23.4- / 21.0
//     a layer's weight gradients, hidden size (x 4) and rows: 768 2048 232 / 166* / 215, 512 68 / 56* / 70; 1024 2048 390 / 268* / 339; 1600 2048
//        955 / 700* / 867; 576 1077 88* / 109-, 2697 192* / 229-; 832 256 57* / 70-; 256 2048 47* / 77 / 55
// Large ones are 1300 TFLOP/s of bf16 on ordinary data, two thirds of what the instruction sustains from registers.  Tried: 64x64 accumulators a wave
// (768x3072 135, 4096 720), 64x64 tiles (76; 840), two blocks a CU of 128x64 (128 registers: 74), all values of a k-tile split at once (4096 690).
PiecesTile pick_pieces(const bb_gemm_desc* descs, int count) {
    struct Estimate {
        double base, outputs, full, first[5], after[5], split[5];     // fp32: us, us per 10^6 outputs; us a k of four tiles, of up to four, of as many behind fours
        struct {
            double base, outputs, round, step, more, share;           // (more: a k of several rounds)
        } tile[2];                                                    // 128x128, 128x64
    };
    static const Estimate products = {4.0, 1.15, 0.0563, {0, 0.0215, 0.0343, 0.0491, 0.0643}, {0, 0.0272, 0.0384, 0.0535, 0.0685}, {0, 0.0122, 0.0195, 0.0263, 0.0335},
                                      {{3.9, 0.76, 3.3, 0.0317, 0.0036, 0.0062}, {2.4, 0.70, 2.9, 0.0216, 0.0020, 0.0026}}};
    static const Estimate wgrad = {3.5, 0.97, 0.0583, {0, 0.0209, 0.0340, 0.0487, 0.0633}, {0, 0.0209, 0.0340, 0.0487, 0.0633}, {}, {{2.7, 0.50, 3.4, 0.0338, 0.0, 0.0051}, {}}};
    // (their column sums' launches in both)
    static const Estimate wgrads = {9.6, 2.21, 0.0595, {0, 0.0225, 0.0374, 0.0515, 0.0653}, {0, 0.0225, 0.0374, 0.0515, 0.0653}, {}, {{7.2, 1.14, 7.6, 0.0360, 0.0, 0.0061}, {}}};
    int64_t tiles[2] = {0, 0}, t64 = 0, t32 = 0;
    double outputs = 0.0;
    int k = 0;
    if (count < 1 || count > GROUP_MAX) return P_NONE;
    for (int i = 0; i < count; ++i) {
        const bb_gemm_desc& d = descs[i];
        if (!d.pieces || d.dtype != BB_F32 || d.nb1 > 1 || d.nb2 > 1 || d.conv_c != 0 || (count > 1 && d.layout != BB_TN)) return P_NONE;
        // vectors of four along every row, and tiles within 32-bit offsets
        if (d.M <= 0 || d.N <= 0 || d.K <= 0 || d.N % 4 || d.ldc % 4 || d.ldaux % 4 || d.lda >= (1 << 21) || d.ldb >= (1 << 21)) return P_NONE;
        for (const void* p : {(const void*)d.C, d.bias, d.aux_in, (const void*)d.aux_out, d.resid})
            if ((uintptr_t)p % 16) return P_NONE;
        auto count_tiles = [&](int m, int n) { return (int64_t)((d.M + m - 1) / m) * ((d.N + n - 1) / n); };
        tiles[0] += count_tiles(128, 128);
        tiles[1] += count_tiles(128, 64);
        t64 += count_tiles(64, 64);
        t32 += count_tiles(64, 32);
        outputs += 1e-6 * d.M * d.N;
        k = d.K > k ? d.K : k;
    }
    if (t64 < 128) return P_NONE;       // (half of the CUs: the fp32 kernels share such a contraction out)
    auto rounds = [](int64_t n) { return (double)((n + 255) / 256); };
    const bool product = descs[0].layout != BB_TN;
    const Estimate& e = product ? products : count == 1 ? wgrad : wgrads;
    const bool split = count == 1 && pick_f32_split(descs[0].M, descs[0].N, descs[0].K, 1, descs[0].layout);
    const int64_t fours = split ? 0 : t64 / 1024, most = ((split ? t32 : t64) - 1024 * fours + 255) / 256;
    const double fp32 = e.base + e.outputs * outputs + (split ? e.split[most] : fours ? fours * e.full + e.after[most] : e.first[most]) * k;
    auto pieces = [&](int t) {
        const double r = rounds(tiles[t]);
        return e.tile[t].base + e.tile[t].outputs * outputs + r * e.tile[t].round + (r * e.tile[t].step + (r > 1 ? e.tile[t].more : 0.0) + e.tile[t].share / 256 * tiles[t]) * k;
    };
    const double large = pieces(0), small = product ? pieces(1) : large, line = (!product ? 0.97 : k < 256 ? 0.95 : 1.0) * fp32;
    if (large < line && large < 1.05 * small) return P128x128;
    return small < line ? P128x64 : P_NONE;
}

template <int TM, int TN, int WM, int WN, bool TA, bool TB> static int launch(GemmArgs& g, hipStream_t st) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16, smem = 2 * 3 * (BM + BN) * 64;
    auto kern = gemm_f32_pieces_kernel<TM, TN, WM, WN, TA, TB>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    bb_launch(kern, dim3(g.tiles_m * g.tiles_n), dim3(WM * WN * 64), smem, st, g);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
int launch_pieces(GemmArgs& g, int layout, PiecesTile tile, hipStream_t st) {
    if (layout == BB_TN) return launch<4, 2, 2, 4, true, true>(g, st);
    if (tile == P128x128) return layout == BB_NT ? launch<4, 2, 2, 4, false, false>(g, st) : launch<4, 2, 2, 4, false, true>(g, st);
    return layout == BB_NT ? launch<2, 2, 4, 2, false, false>(g, st) : launch<2, 2, 4, 2, false, true>(g, st);
}
int launch_pieces_grouped(GroupedArgs& G, hipStream_t st) {
    constexpr int smem = 2 * 3 * 256 * 64;
    auto kern = gemm_f32_pieces_grouped_kernel<4, 2, 2, 4>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, smem));
    int blocks = 0;
    for (int i = 0; i < G.count; ++i) {
        GemmArgs& g = G.p[i];
        g.tiles_m = (g.M + 127) / 128;
        g.tiles_n = (g.N + 127) / 128;
        G.first_block[i] = blocks;
        blocks += g.tiles_m * g.tiles_n;
    }
    G.first_block[G.count] = blocks;
    bb_launch(kern, dim3(G.ride.blocks + blocks), dim3(512), smem, st, G);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
