// bf16 products on v_mfma_f32_16x16x32_bf16: NT and NN products on tiles of 256x256 down to 32x64, and large weight gradients (TN).
//
// Why this instruction: the card's power.  From registers, on normal data, 32x32x16 sustains 1777 TFLOP/s and 16x16x32 2030 (on zeros both
// 2470): per multiplication it moves half the accumulators.  The sums are the same: one 16x16x32 adds its contraction in the order in which
// two 32x32x16 do, so these kernels and those of gemm_kernels.h give equal bits.
//
// What bounds a large product, counted in stages of 1024 and 1600 columns: power a tenth (2.05 to 2.25 of 2.4 GHz); the matrix pipe is 34 to 50 %
// busy, 36 to 62 % of a CU in use.  The rest is CUs without a tile (the last round, 192 tiles of weight gradients), what a tile costs around its
// loop -- 256x256 tiles with two outputs or times a tensor 34 and 37 % --, and waits for LDS and transfers.
//
// Loop: 64-wide k-tiles, global -> LDS by DMA, a ring of STAGES of them, two steps of 32 a k-tile.  While the matrix cores work on one
// step's fragments the other step's are read into a second register set.  One barrier a k-tile: behind it the k-tile's own stage is
// read and the next k-tile has landed, so the transfers of the k-tile STAGES further on go into that stage, spread over the matrix
// instructions that follow.  No branch inside: what changes towards the end of a contraction is done by the loops around the step.
//
// Small tiles (at most about a round of them): such a launch waits for its chain of k-tiles, each a few hundred nanoseconds of LDS latency, barrier
// and transfers with the matrix pipe idle most of the time.  Two things shorten it.  Twice the waves of half the size (16 to 64 rows, 32 columns):
// a SIMD has another wave to go on with.  And WHOLE: fragments are read a whole k-tile ahead, into a second set of registers for both steps; the
// barrier at the head of a k-tile then says that everybody holds it (its stage is free) and that the next one has landed.  Device time, us, kernel
// before (32x32x16, half the waves, a k-tile ahead) / half a k-tile ahead / a whole one: 32x64 tiles NT 1024x512x2048 8.4 / 7.6 / 6.8, x512
// 4.2 / 4.3 / 3.8, NN 8.8 / 8.5 / 6.9; 64x128 NN 2043x768x3072 17.9 / 16.4 / 17.0, 2048x1024x4096 23.9 / 22.0 / 22.9, NT 25.0 / 21.9 / 23.4; 128x64 NT
// 1024x2048x512 with activation 8.2 / 7.1 / 6.8; 128x128 with a residual NT 4096x768x3072 25.1 / 24.5 / 24.0, NN 8192x512x2048 21.8 / - / 20.5.
// Twice the waves on 32x32x16 take half of that (64x128 NN 2043x768x3072 17.4, 2048x1024x4096 23.7); one wave a SIMD half a k-tile ahead is
// twice as slow (64x128 2043x768x3072 32.3).
//
// LDS: rows of a k-contiguous operand are 128 bytes, of a k-major one a k each; 16-byte chunks are swizzled so that the sixteen or
// thirty-two lanes LDS serves at a time fall on different banks (counted: none conflicts, but of NN's B, whose two groups of sixteen lanes, eight k
// apart, meet on the same half of their chunks: conflicts are a quarter, of 256x128 tiles a third of LDS' cycles, LDS 19 and 38 % busy).  The product is made
// transposed (B times A): a lane holds one row of C.  NT and NN read the columns of two neighbouring fragments interleaved, so that its two accumulators are
// eight neighbouring columns and a store is 16 bytes; weight gradients store fp32, where four columns are.
#pragma once
#include "gemm_kernels.h"

__device__ __forceinline__ const char* m16_uniform(const char* p) {
    const uint64_t b = (uint64_t)p;
    return (const char*)(((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b));
}
// the same value, made anew where this stands: the compiler computes what depends on it only there, not in front of the loops, where it
// would lie in registers that the fragments need (256x256 tiles: none spills, and one that did inside the loop would be a wait for every transfer)
__device__ __forceinline__ int m16_here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
// chunk swizzle of a k-contiguous tile by its row.  A fragment's sixteen rows are neighbours, or (PAIRED) four groups of four, eight apart
template <bool PAIRED> __host__ __device__ constexpr int m16_row_swizzle(int r) { return PAIRED ? ((r >> 1) & 1) | (((r >> 3) & 3) << 1) : (r >> 1) & 7; }
// ... and of a k-major tile by its k: the four k of a transposing read (two chunks each, PAIRED four) on different banks -- as far as rows
// of BR * 2 bytes do not see to that themselves --, then those of two groups of sixteen lanes, eight k apart
template <int BR, bool PAIRED> __host__ __device__ constexpr int m16_k_swizzle(int k) {
    const int four = BR % 128 == 0 ? 4 * (k & 3) : BR % 64 == 0 ? 4 * ((k >> 1) & 1) : 0;
    return PAIRED ? four : four ^ (((k >> 3) & 1) << 1);
}

// A wave's transfers of one operand tile, BR rows (columns of a k-major operand) x 64 k: base in scalar registers, a 32-bit offset per lane
// and transfer (leading dimensions below kDmaMaxLd).
template <int BR, int NW, bool KM, bool PAIRED> struct M16Lanes {
    static constexpr int BYTES = BR * 128, PIECES = BYTES / 1024, ROUNDS = (PIECES + NW - 1) / NW, CPR = BR / 8;
    static_assert(BR % 32 == 0, "whole transfers");
    const char* base;
    int64_t step;      // bytes per k-tile
    unsigned off[ROUNDS];

    __device__ __forceinline__ void init(const bf16* at, int64_t ld, int row0, int rows, int tid) {
        const int ld2 = (int)ld * 2;
        if constexpr (!KM) {
            const int r0 = tid >> 3, last = rows - 1 - row0;
            const int c = (tid & 7) ^ m16_row_swizzle<PAIRED>(r0);
            static_assert(NW * 8 % 32 == 0, "a round later the chunks lie as in the round before");
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i) off[i] = __umul24((unsigned)min(r0 + i * (NW * 8), last), (unsigned)ld2) + c * 16;
            base = (const char*)(at + (int64_t)row0 * ld);
            step = 128;
        } else {
            reach(ld2, rows - 8 - row0, tid, 64);
            base = (const char*)(at + row0);
            step = 128 * ld;
        }
    }
    // (left: KM only, k rows the tile has; a lane past them reads the last one again)
    __device__ __forceinline__ void reach(int ld2, int last, int tid, int left) {
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int q = i * NW * 64 + tid, k = q / CPR, c = (q - k * CPR) ^ m16_k_swizzle<BR, PAIRED>(k);
            off[i] = __umul24((unsigned)min(k, left - 1), (unsigned)ld2) + min(c * 8, last) * 2;
        }
    }
    // (live 0: nothing is moved, but the transfer counts; so do those of a wave that the last round has no piece for)
    template <int I> __device__ __forceinline__ void issue(unsigned tile, int wave, int live) {
        if constexpr (I == 0) base = m16_uniform(base);
        if constexpr (PIECES % NW != 0 && I == ROUNDS - 1) live = I * NW + wave < PIECES ? live : 0;
        dma16_base_masked(base, off[I], tile + (I * NW + wave) * 1024, __builtin_amdgcn_readfirstlane(live));
        if constexpr (I == ROUNDS - 1) base += step;
    }
};

// a wave's fragments, T of 16 rows x 32 k, from tile row (column) wbase on; lane l holds row l % 16, k = 8 (l / 16) .. + 7.
// KM: fragment t is the one numbered place(t, first) behind wbase.  Where T is a power of two, so is the number of chunks a wave spans, and
// a fragment's offset is that of the first one with some bits turned: one register instead of T, one v_xad_u32 a read.
template <int BR, int T, bool KM, bool PAIRED> struct M16Frags {
    static constexpr bool TURN = (T & (T - 1)) == 0 && BR % 128 == 0;
    static constexpr int EACH = PAIRED ? 32 : 16, COUNT = PAIRED ? T / 2 : T;   // columns and number of what shares an offset
    int off[KM ? (TURN ? 1 : COUNT) : 2];
    static __device__ __forceinline__ int place(int t, int first) { return TURN ? t ^ first : t + first < T ? t + first : t + first - T; }
    __device__ __forceinline__ void init(int wbase, int lane, int first = 0) {
        if constexpr (!KM) {
            const int i = lane & 15, row = wbase + (PAIRED ? 8 * (i >> 2) + (i & 3) : i);
            off[0] = row * 128 + (((lane >> 4) ^ m16_row_swizzle<PAIRED>(row)) << 4);
            off[1] = off[0] ^ 64;
        } else {
            const int j = lane & 15, k = (lane >> 4) * 8 + (j >> 2);
#pragma unroll
            for (int t = 0; t < (TURN ? 1 : COUNT); ++t) {
                const int chunk = ((wbase + place(t, first) * EACH) >> 3) + (PAIRED ? (j & 3) : ((j & 3) >> 1));
                off[t] = k * (BR * 2) + ((chunk ^ m16_k_swizzle<BR, PAIRED>(k)) << 4) + (PAIRED ? 0 : (j & 1) * 8);
            }
        }
    }
    // (at the head of a step: the reads' offsets are made where they are, not held)
    __device__ __forceinline__ void here() {
        if constexpr (KM && TURN) off[0] = m16_here(off[0]);
    }
    __device__ __forceinline__ bf16x8 load(const unsigned char* tile, int t, int ks) const {
        if constexpr (!KM) {
            return *(const bf16x8*)(tile + off[ks] + (PAIRED ? (t >> 1) * 4096 + (t & 1) * 512 : t * 2048));
        } else {
            const int n = PAIRED ? t >> 1 : t;
            const unsigned char* p = tile + (TURN ? off[0] ^ (n * EACH * 2) : off[TURN ? 0 : n]) + (PAIRED ? (t & 1) * 8 : 0) + ks * 32 * (BR * 2);
            typedef __attribute__((ext_vector_type(8))) short s16x8;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 4 * (BR * 2)));
            return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

// The tile's accumulators, its place in the ring, and the step over one k-tile.
template <int TM, int TN, int WM, int WN, bool AKM, bool BKM, bool PAIRED, int STAGES, bool WHOLE = false> struct M16Loop {
    static constexpr int NW = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16;
    using OpA = M16Lanes<BM, NW, AKM, false>;
    using OpB = M16Lanes<BN, NW, BKM, PAIRED>;
    using FragA = M16Frags<BM, TM, AKM, false>;
    static constexpr int STAGE_BYTES = OpA::BYTES + OpB::BYTES, LOADS = OpA::ROUNDS + OpB::ROUNDS;
    static constexpr int NM = TM * TN, NF = TM + TN;
    // ROWS: the registers of A's fragments are filled again row by row, each when the row's products have gone out, instead of a second set:
    // 32 registers of 256x256 tiles, which spill without.  The barrier then stands in the second step, WAIT instructions down (a read's
    // latency behind the first step's last), the transfers in what is left of it.  Else the first half of a step carries the reads, the barrier
    // stands in the first step, five eighths down, the transfers behind it over as many instructions as a step has.
    static constexpr bool ROWS = TM >= 8;
    static constexpr int WAIT = 2 * TN;
    static constexpr int READS = NM / 2, BARRIER = ROWS ? NM + WAIT : NM * 5 / 8, FEEDS = ROWS ? NM - WAIT : NM;
    OpA opa;
    OpB opb;
    FragA fa;
    M16Frags<BN, TN, BKM, PAIRED> fb;
    f32x4 acc[TM][TN];
    static constexpr int SETS = WHOLE ? 4 : 2;     // one a step of the k-tiles whose fragments are held
    static_assert(!ROWS || !WHOLE, "one set of rows, half a k-tile ahead");
    bf16x8 a[ROWS ? 1 : SETS][TM], b[SETS][TN];
    float sum, part;
    int wave, stage, first;
    unsigned lds0;
    unsigned char* smem;

    // (first_fragment: KM, of the wave's fragments of A the one it starts with)
    __device__ __forceinline__ void init(unsigned char* lds, int tid, int first_fragment = 0) {
        smem = lds;
        lds0 = (unsigned)(uintptr_t)(lds_ptr_t*)lds;
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        stage = 0;
        first = first_fragment;
        fa.init(wave / WN * (TM * 16), tid & 63, first);
        fb.init(wave % WN * (TN * 16), tid & 63);
    }
    template <int I> __device__ __forceinline__ void feed(unsigned at, int live) {
        if constexpr (I < OpA::ROUNDS) opa.template issue<I>(at, wave, live);
        else opb.template issue<I - OpA::ROUNDS>(at + OpA::BYTES, wave, live);
    }
    __device__ __forceinline__ void feed_all(int t, int live) {
        static_for([&](auto i) { feed<decltype(i)::value>(lds0 + t * STAGE_BYTES, live); }, std::make_integer_sequence<int, LOADS>{});
    }
    // step ks's fragments in the order of their use (SET: WHOLE, which k-tile's registers)
    template <int Q, int SET = 0> __device__ __forceinline__ void read(const unsigned char* st, int ks) {
        const int s = ROWS ? 0 : 2 * SET + ks;
        if constexpr (Q == 0) a[s][0] = fa.load(st, 0, ks);
        else if constexpr (Q <= TN) b[2 * SET + ks][Q - 1] = fb.load(st + OpA::BYTES, Q - 1, ks);
        else a[s][Q - TN] = fa.load(st, Q - TN, ks);
    }
    __device__ __forceinline__ void read_first() {
        static_for([&](auto q) { read<decltype(q)::value % NF>(smem + stage * STAGE_BYTES, decltype(q)::value / NF); },
                   std::make_integer_sequence<int, WHOLE ? 2 * NF : NF>{});
    }
    template <int NEWER> __device__ __forceinline__ void landed() {   // all but the NEWER latest k-tiles of this wave; then everybody's
        asm volatile("" ::: "memory");
        wait_vmcnt_lgkm0<NEWER * LOADS>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        sum = 0.f;
    }
    // SUMS: the wave adds up the k of its first fragment of A, a few beside each product of the row (at once they would hold up the next one).
    // One k-tile: multiplied, its second step's and the next k-tile's first fragments read, the k-tile STAGES on sent for (live -1).
    template <bool SUMS = false> __device__ __forceinline__ void step(int live) {
        fa.here();
        fb.here();
        const unsigned char* cur = smem + stage * STAGE_BYTES;
        const unsigned into = lds0 + stage * STAGE_BYTES;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        const unsigned char* nxt = smem + stage * STAGE_BYTES;
        static_for(
            [&](auto idx) {
                constexpr int m = decltype(idx)::value, s = m / NM, mm = m % NM, i = mm / TN, j = mm % TN;
                if constexpr (m == BARRIER) landed<STAGES - 2>();
                const bf16x8& row = a[ROWS ? 0 : s][i];
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][j], row, acc[i][j], 0, 0, 0);
                if constexpr (SUMS && i == 0) {
                    if constexpr (j == 0) part = 0.f;
#pragma unroll
                    for (int e = 8 * j / TN; e < 8 * (j + 1) / TN; ++e) part += (float)row[e];
                    if constexpr (j == TN - 1) {
                        typedef __attribute__((ext_vector_type(2))) unsigned u2;
                        const u2 both = __builtin_bit_cast(u2, __builtin_amdgcn_permlane32_swap(__float_as_uint(part), __float_as_uint(part), false, false));
                        sum += __uint_as_float(both[0]);
                        sum += __uint_as_float(both[1]);
                    }
                }
                if constexpr (m >= BARRIER && m < BARRIER + FEEDS)
                    static_for([&](auto d) { feed<LOADS * (m - BARRIER) / FEEDS + decltype(d)::value>(into, live); },
                               std::make_integer_sequence<int, LOADS * (m - BARRIER + 1) / FEEDS - LOADS * (m - BARRIER) / FEEDS>{});
                const unsigned char* src = s == 0 ? cur : nxt;
                if constexpr (ROWS) {
                    __builtin_amdgcn_sched_barrier(0);     // (a read in front of the row's last product would need registers of its own)
                    constexpr int first = s == 0 ? 0 : WAIT;      // from here on the next step's fragments may be read
                    if constexpr (mm >= first && mm < first + TN) read<1 + mm - first>(src, 1 - s);
                    if constexpr (mm >= first && mm < first + first / TN) a[0][mm - first] = fa.load(src, mm - first, 1 - s);
                    if constexpr (mm >= first && j == TN - 1) a[0][i] = fa.load(src, i, 1 - s);
                } else if constexpr (mm < READS) {
                    static_for([&](auto d) { read<NF * mm / READS + decltype(d)::value>(src, 1 - s); },
                               std::make_integer_sequence<int, NF * (mm + 1) / READS - NF * mm / READS>{});
                }
                __builtin_amdgcn_sched_barrier(0);
            },
            std::make_integer_sequence<int, 2 * NM>{});
    }
    // WHOLE: one k-tile out of the registers SET, the next one's fragments into the others beside three quarters of its products (what is left
    // covers the last reads), the transfers of the k-tile STAGES on, into this one's stage, beside all of them.  Behind the last k-tile the
    // reads bring what nothing uses.
    template <int SET> __device__ __forceinline__ void step_whole(int live) {
        constexpr int CARRY = 2 * NM - (NM + 1) / 2;
        const unsigned into = lds0 + stage * STAGE_BYTES;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        const unsigned char* nxt = smem + stage * STAGE_BYTES;
        landed<STAGES - 2>();
        static_for(
            [&](auto idx) {
                constexpr int m = decltype(idx)::value, s = 2 * SET + m / NM, i = m % NM / TN, j = m % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][j], a[s][i], acc[i][j], 0, 0, 0);
                if constexpr (m < CARRY)
                    static_for(
                        [&](auto d) {
                            constexpr int q = 2 * NF * m / CARRY + decltype(d)::value;
                            read<q % NF, 1 - SET>(nxt, q / NF);
                        },
                        std::make_integer_sequence<int, 2 * NF * (m + 1) / CARRY - 2 * NF * m / CARRY>{});
                static_for([&](auto d) { feed<LOADS * m / (2 * NM) + decltype(d)::value>(into, live); },
                           std::make_integer_sequence<int, LOADS * (m + 1) / (2 * NM) - LOADS * m / (2 * NM)>{});
                __builtin_amdgcn_sched_barrier(0);
            },
            std::make_integer_sequence<int, 2 * NM>{});
    }
};

// the tiles that store fp32, too (larger ones have no registers left for it)
template <int TM, int TN> constexpr bool kM16F32Out = TM * TN <= 16;

// NT and NN products over whole k-tiles.  A block walks the tiles b, b + gridDim.x, ... (a multiple of 8 apart, so that they stay on its XCD, or
// one tile a block): the next tile's first k-tiles go out under the last of this one and land under its epilogue.  More than one tile
// a block needs K >= STAGES * 64: the waits count on a tile's transfers filling the ring.  WHOLE: one tile a block.
template <int TM, int TN, int WM, int WN, bool BKM, int STAGES, bool WHOLE, bool DROP>
__global__ __launch_bounds__(WM* WN * 64) void gemm_bf16_m16_kernel(const GemmArgs g) {
    using Loop = M16Loop<TM, TN, WM, WN, false, BKM, true, STAGES, WHOLE>;
    constexpr int BM = Loop::BM, BN = Loop::BN, NP = TN / 2;
    static_assert(TN % 2 == 0, "fragments in pairs");
    constexpr int GROUP_M = BM == 256 && BN < 256 ? 4 : 8;   // (32 tiles of an XCD: 4 x 8 of 256 x 128 read fewer rows than 8 x 4)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // what leads to the first transfer, fetched together (see gemm_bf16_dma_body)
    asm volatile("" ::"s"(g.A), "s"(g.B), "s"(g.lda), "s"(g.ldb), "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.tiles_m), "s"(g.tiles_n));
    const int tid = threadIdx.x, total = g.tiles_m * g.tiles_n, G = gridDim.x, KT = g.K / 64;
    const bf16* A = (const bf16*)g.A;
    const bf16* B = (const bf16*)g.B;
    int64_t coff = 0;
    if (blockIdx.z != 0) {
        const int b1 = blockIdx.z / g.nb2, b2 = blockIdx.z % g.nb2;
        A += b1 * g.sA1 + b2 * g.sA2;
        B += b1 * g.sB1 + b2 * g.sB2;
        coff = b1 * g.sC1 + b2 * g.sC2;
    }
    Loop p;
    int tile = blockIdx.x, tm, tn;
    auto point_at = [&](int m, int n) {
        const int t = m16_here(tid);
        p.opa.init(A, g.lda, m * BM, g.M, t);
        p.opb.init(B, g.ldb, n * BN, g.N, t);
    };
    tile_coords<GROUP_M>(tile, g.tiles_m, g.tiles_n, tm, tn);
    point_at(tm, tn);
    p.init(smem, tid);
#pragma unroll
    for (int t = 0; t < STAGES; ++t) p.feed_all(t, __builtin_amdgcn_readfirstlane((t - KT) >> 31));
    p.template landed<STAGES - 1>();
    for (;;) {
        p.clear();
        p.read_first();
        if constexpr (WHOLE) {
            auto live_at = [&](int kt) { return __builtin_amdgcn_readfirstlane((kt + STAGES - KT) >> 31); };
            int kt = 0;
            for (; kt + 1 < KT; kt += 2) {
                p.template step_whole<0>(live_at(kt));
                p.template step_whole<1>(live_at(kt + 1));
            }
            if (kt < KT) p.template step_whole<0>(0);
        } else {
            for (int kt = STAGES; kt < KT; ++kt) p.step(-1);
        }
        const int next = tile + G, live = WHOLE ? 0 : __builtin_amdgcn_readfirstlane((next - total) >> 31);
        int next_m = 0, next_n = 0;
        if (live) {
            tile_coords<GROUP_M>(next, g.tiles_m, g.tiles_n, next_m, next_n);
            point_at(next_m, next_n);
        }
        if constexpr (!WHOLE)
            for (int t = min(KT, STAGES); t > 0; --t) p.step(live);

        // Epilogue from the registers: the lane's row of 16 row groups, eight columns of each pair of fragments.  The operand of the kinds
        // that read one is fetched AHEAD row groups before its use, the pieces of a row are made first and stored one behind the
        // other.  Lanes outside the matrix read inside it and store nothing.
        const int lane = m16_here(tid) & 63;
        const int row = tm * BM + p.wave / WN * (TM * 16) + (lane & 15), col = tn * BN + p.wave % WN * (TN * 16) + 8 * (lane >> 4);
        u32x4 bias[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q)
            if (g.bias) bias[q] = *(const u32x4*)((const bf16*)g.bias + min(col + q * 32, g.N - 8));
        auto finish = [&](auto kind_c, auto held_c) {
            constexpr int kind = decltype(kind_c)::value, AHEAD = TM > 4 ? 2 : TM;
            constexpr bool HELD = decltype(held_c)::value;
            constexpr bool READS = kind == BB_EPI_DACT || kind == BB_EPI_RESIDUAL || kind == BB_EPI_MUL || kind == BB_EPI_MUL_POS || kind < 0;
            const bf16* operand = kind < 0 ? epilogue_operand(g) : (const bf16*)(kind == BB_EPI_RESIDUAL ? g.resid : g.aux_in);
            u32x4 op[AHEAD][NP];
            auto fetch = [&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                if (!READS || (kind < 0 && !operand)) return;
                const bf16* r = operand + coff + (int64_t)min(row + i * 16, g.M - 1) * g.ldaux;
#pragma unroll
                for (int q = 0; q < NP; ++q) op[i % AHEAD][q] = *(const u32x4*)(r + min(col + q * 32, g.N - 8));
            };
            static_for([&](auto i_c) { fetch(i_c); }, std::make_integer_sequence<int, AHEAD>{});
            static_for(
                [&](auto i_c) {
                    constexpr int i = decltype(i_c)::value;
                    const int m = row + i * 16, mc = min(m, g.M - 1);
                    const int64_t ci = coff + (int64_t)m * g.ldc + col, xi = coff + (int64_t)m * g.ldaux + col;
                    HeldStore held[NP];
                    static_for(
                        [&](auto q_c) {
                            constexpr int q = decltype(q_c)::value;
                            float v[8], b8[8];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                v[e] = p.acc[i][2 * q][e];
                                v[4 + e] = p.acc[i][2 * q + 1][e];
                            }
                            if (g.alpha != 1.0f) {
#pragma unroll
                                for (int e = 0; e < 8; ++e) v[e] *= g.alpha;
                            }
                            if (g.bias) unpack_bf16x8(bias[q], b8);
                            const int n = col + q * 32, nc = HELD ? min(n, g.N - 8) : n;
                            const int64_t xr = HELD ? coff + (int64_t)mc * g.ldaux + nc : xi + q * 32;
                            if (HELD || (m < g.M && n < g.N))
                                epilogue_vec8_at<DROP, true, false, false, kind, HELD>(g, ci + q * 32, xr, HELD ? mc : m, nc, v, b8, op[i % AHEAD][q],
                                                                                       u32x4{0u, 0u, 0u, 0u}, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}, &held[q]);
                        },
                        std::make_integer_sequence<int, NP>{});
                    if constexpr (i + AHEAD < TM) fetch(std::integral_constant<int, i + AHEAD>{});
                    if constexpr (HELD) {
                        if (m < g.M) {
#pragma unroll
                            for (int q = 0; q < NP; ++q)
                                if (col + q * 32 < g.N) *(u32x4*)((bf16*)g.C + ci + q * 32) = held[q].c;
                            if (kind == BB_EPI_ACT_DACT || (kind == BB_EPI_ACT && g.aux_out)) {
#pragma unroll
                                for (int q = 0; q < NP; ++q)
                                    if (col + q * 32 < g.N) *(u32x4*)((bf16*)g.aux_out + xi + q * 32) = held[q].aux;
                            }
                        }
                    }
                },
                std::make_integer_sequence<int, TM>{});
        };
        if (kM16F32Out<TM, TN> && g.c_f32) {
            if constexpr (kM16F32Out<TM, TN>) finish(std::integral_constant<int, -1>{}, std::false_type{});
        } else {
            switch (g.epilogue) {
                case BB_EPI_ACT: finish(std::integral_constant<int, BB_EPI_ACT>{}, std::true_type{}); break;
                case BB_EPI_DACT: finish(std::integral_constant<int, BB_EPI_DACT>{}, std::true_type{}); break;
                case BB_EPI_RESIDUAL: finish(std::integral_constant<int, BB_EPI_RESIDUAL>{}, std::true_type{}); break;
                case BB_EPI_MUL: finish(std::integral_constant<int, BB_EPI_MUL>{}, std::true_type{}); break;
                case BB_EPI_MUL_POS: finish(std::integral_constant<int, BB_EPI_MUL_POS>{}, std::true_type{}); break;
                case BB_EPI_ACT_DACT: finish(std::integral_constant<int, BB_EPI_ACT_DACT>{}, std::true_type{}); break;
                default: finish(std::integral_constant<int, BB_EPI_NONE>{}, std::true_type{}); break;
            }
        }
        if (!live) return;
        tile = next;
        tm = next_m;
        tn = next_n;
    }
}

// Weight gradients: C[m][n] (fp32) = or += alpha * sum over k of A[k][m] B[k][n], both operands k-major, K > STAGES * 64.
//
// A last k-tile that is not whole: its transfers read the last row again (nothing lies behind it), and once they have landed the rows
// past the end are cleared in LDS, in both operands, before they are read.
//
// Column sums of A (a bias gradient): the waves of a row of waves, in the blocks of the first tile columns, hold the same fragments of A; each
// starts with another and adds that one up beside its products.  (By its number in the code: nothing is chosen inside the loop.  One fragment a
// wave: with two, in the first column alone, the blocks of that column took a tenth longer, and a launch of one round with them.)  Per 32 k a lane
// adds its eight, then (the lower half of the wave) what the lane 32 further on has; the two chains of a row are put together at the end.
// That is the order of gemm_bf16_dma_body, whose lanes add eight of sixteen k a step.
constexpr int m16_sum_columns(int TM, int WN) { return (TM + WN - 1) / WN; }   // tile columns that takes: a problem with sums has as many
template <int TM, int TN, int WM, int WN, int STAGES>
__device__ __forceinline__ void wgrad_m16_body(const GemmArgs& g, const int id) {
    using Loop = M16Loop<TM, TN, WM, WN, true, true, false, STAGES>;
    constexpr int BM = Loop::BM, BN = Loop::BN, NT = Loop::NW * 64;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x;
    const int KT = (g.K + 63) / 64, tail = g.K & 63;
    int tm, tn;
    panel_coords<8>(id, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    Loop p;
    p.opa.init((const bf16*)g.A, g.lda, m0, g.M, tid);
    p.opb.init((const bf16*)g.B, g.ldb, n0, g.N, tid);
    constexpr int SC = m16_sum_columns(TM, WN);
    const int first = __builtin_amdgcn_readfirstlane((tid >> 6) % WN * SC + tn);
    const bool do_sums = g.colsum != nullptr && tn < SC && first < TM;
    p.init(smem, tid, do_sums ? first : 0);
    auto last_tile = [&]() {     // the transfers that go out next are those of the last k-tile
        if (!tail) return;
        const int t = m16_here(tid);
        p.opa.reach((int)g.lda * 2, g.M - 8 - m0, t, tail);
        p.opb.reach((int)g.ldb * 2, g.N - 8 - n0, t, tail);
    };
    p.clear();
#pragma unroll
    for (int t = 0; t < STAGES; ++t) p.feed_all(t, -1);
    p.template landed<STAGES - 1>();

    const int wm = p.wave / WN, wn = p.wave % WN;
    auto walk = [&](auto sums_c) {
        constexpr bool SUMS = decltype(sums_c)::value;
        p.read_first();
        int kt = 0;
        for (const int whole = KT - (tail ? 1 : 0); kt + STAGES < whole; ++kt) p.template step<SUMS>(-1);
        for (; kt < KT; ++kt) {
            if (tail && kt + STAGES == KT - 1) last_tile();
            if (tail && kt == KT - 1) {
                // everything has landed (the ring holds nothing behind it), no wave reads on before the rows are cleared
                p.template landed<0>();
                const int t = m16_here(tid);
                unsigned char* st = smem + p.stage * Loop::STAGE_BYTES;
                for (int b = tail * BM * 2 + t * 16; b < Loop::OpA::BYTES; b += NT * 16) *(u32x4*)(st + b) = u32x4{0u, 0u, 0u, 0u};
                for (int b = tail * BN * 2 + t * 16; b < Loop::OpB::BYTES; b += NT * 16) *(u32x4*)(st + Loop::OpA::BYTES + b) = u32x4{0u, 0u, 0u, 0u};
                p.template landed<0>();
                p.read_first();
            }
            p.template step<SUMS>(__builtin_amdgcn_readfirstlane((kt + STAGES - KT) >> 31));
        }
    };
    if (do_sums) walk(std::true_type{});
    else walk(std::false_type{});
    const int lane = m16_here(tid) & 63;
    if (do_sums) {
        const float t = p.sum + __shfl_xor(p.sum, 16, 64);
        const int m = m0 + (wm * TM + first) * 16 + (lane & 15);
        if (lane < 16 && m < g.M) g.colsum[m] += t;
    }

    const int row0 = m0 + wm * (TM * 16) + (lane & 15), col = n0 + wn * (TN * 16) + 4 * (lane >> 4);
    auto row = [&](int i) { return row0 + Loop::FragA::place(i, p.first) * 16; };
    constexpr int AHEAD = TM > 4 ? 2 : TM;
    f32x4 old[AHEAD][TN];
    auto fetch = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        if (!g.accumulate) return;
        const float* c = (const float*)g.C + (int64_t)min(row(i), g.M - 1) * g.ldc;
#pragma unroll
        for (int j = 0; j < TN; ++j) old[i % AHEAD][j] = *(const f32x4*)(c + min(col + j * 16, g.N - 4));
    };
    static_for([&](auto i_c) { fetch(i_c); }, std::make_integer_sequence<int, AHEAD>{});
    static_for(
        [&](auto i_c) {
            constexpr int i = decltype(i_c)::value;
            const int m = row(i);
            float* c = (float*)g.C + (int64_t)m * g.ldc + col;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 v = p.acc[i][j] * g.alpha;
                if (g.accumulate) v = old[i % AHEAD][j] + v;
                if (m < g.M && col + j * 16 < g.N) *(f32x4*)(c + j * 16) = v;
            }
            if constexpr (i + AHEAD < TM) fetch(std::integral_constant<int, i + AHEAD>{});
        },
        std::make_integer_sequence<int, TM>{});
}
// a layer's in one launch (the tiles of all problems one list, see gemm_bf16_dma_grouped_kernel); two waves a SIMD
template <int TM, int TN, int WM, int WN, int STAGES> __global__ __launch_bounds__(WM* WN * 64, 2) void wgrad_m16_grouped_kernel(const GroupedArgs G) {
    const int id = grouped_place<WM * WN>(G);
    if (id < 0) return;
    int pi = 0;
    while (pi + 1 < G.count && id >= G.first_block[pi + 1]) ++pi;
    wgrad_m16_body<TM, TN, WM, WN, STAGES>(G.p[pi], id - G.first_block[pi]);
}
