// Fused masked softmax-attention for gfx950, bf16, head dimension 64, 32 or 128: forward and the two
// backward kernels (dK/dV and dQ).  No scores or probabilities reach HBM; the forward keeps one fp32
// log-sum-exp per (batch, head, query) for the backward, and, if given room for it, a bit per dropout decision.
//
// Stands in for MultiHeadedAttention.attention of the reference
// (DeepSpeedExamples/pipeline_parallelism/transformer.py:117-127: softmax(QK^T/sqrt(d) with
// masked_fill(mask == 0, -1e9)) V) and for its autograd backward.
//
// Layout.  Q, K, V of head j are the 64-wide column slices at j*64 of the three thirds of the
// [rows, 3*hidden] projection buffer; the context goes to columns j*64 of a [rows, hidden]
// buffer.  Each wave owns 32 rows (queries in forward / dQ, keys in dK/dV) and keeps one score
// COLUMN per lane: scores are produced transposed (S^T = K Q^T), so the softmax reductions over
// keys are in-lane plus one cross-half shuffle, and P^T comes out of the accumulators already
// in the register layout the next MFMA wants as its B operand.  With 32-wide heads (HP = 2) a block
// owns a PAIR of neighbouring heads, whose columns together are one 64-wide slice: the tiles in LDS and
// their loads are those of one 64-wide head, each head has waves of its own, which take the k-steps
// (scores) and the output tile (context, gradients) of that head.  (Waves that took one head after the
// other: 8 x 8 pairs, 128 keys, dropout 9.1 us forward; so, two waves a head, 6.6.)
// Operands that are contracted
// over their row index (V in O = PV, Q and dO in dK/dV, K in dQ) are read from LDS with
// ds_read_b64_tr_b16.  Tiles travel global -> LDS by DMA (global_load_lds_dwordx4),
// double-buffered.  All reductions have a fixed order: results are reproducible bit for bit.
#include "common.h"

#include <type_traits>

typedef __attribute__((address_space(3))) void lds_ptr_t;
typedef const __attribute__((address_space(1))) void gbl_ptr_t;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

struct AttnArgs {
    const bf16* q; const bf16* k; const bf16* v;   // head 0 of batch 0; row stride ld_qkv
    const bf16* o; const bf16* d_o;                // [rows, hidden] context and its gradient
    bf16* out;                                     // forward: context
    bf16* dq; bf16* dk; bf16* dv;                  // backward outputs, row stride ld_dqkv
    float* lse;                                    // [batch, heads, seq], log2 domain
    float* delta;                                  // [batch, heads, seq], rowsum(dO * O)
    const int32_t* key_len;
    uint32_t* keep;                                // dropout: the decisions of the forward (keep_words), or null
    int64_t ld_qkv, ld_o, ld_dqkv;
    int batch, heads, seq, mask;
    float scale_log2;                              // log2(e) / sqrt(d)
    float scale;                                   // 1 / sqrt(d)
    DropKey drop;                                  // dropout on the probabilities (thresh 0: none)
};
template <> struct BbDropAt<AttnArgs> { static constexpr int32_t value = offsetof(AttnArgs, drop); };
template <> struct BbPointersAt<AttnArgs> : BbPointerRun<13> {};   // q .. keep
static_assert(offsetof(AttnArgs, ld_qkv) == 13 * sizeof(void*), "BbPointersAt<AttnArgs>");
// index of probability (b, head, q, kv) in the [batch, heads, seq, seq] tensor that is never stored
__device__ __forceinline__ uint64_t prob_index(const AttnArgs& a, int b, int head, int q) {
    return ((uint64_t)(b * a.heads + head) * a.seq + q) * a.seq;
}

// Global -> LDS transfers (16 or 4 bytes per lane; the LDS target is M0 + lane * size), issued as
// inline assembly: while the compiler sees such a load in flight it turns every wait for an LDS
// read into lgkmcnt(0).  Unseen, fragment waits keep their exact counts; the kernels wait for
// these loads explicitly (wait_vm) before each barrier, as they always did.
// (wave-uniform base, a byte offset per lane)
__device__ __forceinline__ void dma16(const void* base, uint32_t off, const unsigned char* lds_dst) {
    const unsigned m0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_ptr_t*)lds_dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(base) : "m0");
}
__device__ __forceinline__ void dma4(const void* src, const unsigned char* lds_dst) {
    const unsigned m0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_ptr_t*)lds_dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(m0), "v"(src) : "m0");
}

// ---- LDS tile format: [rows][64] bf16, 128 B per row, 16-byte chunk c of row r at slot c ^ fsw(r)
__device__ __forceinline__ int fsw(int r) { return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1); }

// Whole 64-row tile by W waves, eight rows an instruction: row groups wave, wave + W, ...  A wave-uniform base plus the lane's
// offset in bytes (leading dimensions below 2^24: 63 rows fit 32 bits), which only a tile that reaches past the last row clamps.
template <int W> struct LaneOff { uint32_t o[8 / W]; };
template <int W> __device__ __forceinline__ uint32_t lane_row(int i, int wave, int lane) { return (wave + i * W) * 8 + (lane >> 3); }
template <int W> __device__ __forceinline__ LaneOff<W> lane_off(int64_t ld, int wave, int lane) {
    LaneOff<W> l;
#pragma unroll
    for (int i = 0; i < 8 / W; ++i) {
        const uint32_t r = lane_row<W>(i, wave, lane);
        l.o[i] = (r * (uint32_t)ld + (((lane & 7) ^ fsw(r)) << 3)) * 2;
    }
    return l;
}
template <int W>
__device__ __forceinline__ void dma_tile64(const bf16* gbase, int64_t ld, int row0, int last_row, unsigned char* tile,
                                           int wave, int lane, const LaneOff<W>& lo) {
    const bf16* g = gbase + (int64_t)row0 * ld;
    if (row0 + 63 <= last_row) {
#pragma unroll
        for (int i = 0; i < 8 / W; ++i) dma16(g, lo.o[i], tile + (wave + i * W) * 1024);
    } else {
#pragma unroll
        for (int i = 0; i < 8 / W; ++i) {
            const uint32_t r = lane_row<W>(i, wave, lane), past = max((int)r - (last_row - row0), 0);
            dma16(g, lo.o[i] - past * (uint32_t)ld * 2, tile + (wave + i * W) * 1024);
        }
    }
}
// 4-byte variant for the per-row fp32 statistics: 64 consecutive floats
__device__ __forceinline__ void dma_f32x64(const float* gbase, int idx0, int last, unsigned char* dst, int lane) {
    const int i = min(idx0 + lane, last);
    dma4(gbase + i, dst);
}

// A/B fragment along the contiguous (feature) dimension: lane (r = lane%32, kg = lane/32) gets
// features ks*16 + kg*8 .. +8 of tile row row0 + r
__device__ __forceinline__ bf16x8 frag_kc(const unsigned char* tile, int row0, int ks, int lane) {
    const int r = row0 + (lane & 31);
    const int chunk = ks * 2 + (lane >> 5);
    return *(const bf16x8*)(tile + r * 128 + ((chunk ^ fsw(r)) << 4));
}
// A fragment contracted over tile ROWS: lane (c = lane%32, kg = lane/32) gets, for feature column
// col0 + c, the rows rbase + 4kg + {0..3} and rbase + 8 + 4kg + {0..3}: the row order in which a
// 32x32 accumulator column sits in registers 0..7 of a lane
__device__ __forceinline__ bf16x8 frag_tr(const unsigned char* tile, int rbase, int col0, int lane) {
    const int j = lane & 15;
    const int col = col0 + ((lane >> 4) & 1) * 16 + 4 * (j & 3);
    const int r0 = rbase + 4 * (lane >> 5) + (j >> 2);
    const int r1 = r0 + 8;
    const unsigned char* p0 = tile + r0 * 128 + (((col >> 3) ^ fsw(r0)) << 4) + (col & 7) * 2;
    const unsigned char* p1 = tile + r1 * 128 + (((col >> 3) ^ fsw(r1)) << 4) + (col & 7) * 2;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p0);
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p1);
    s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
}
// registers 8*half .. 8*half+7 of a 32x32 accumulator as a bf16 B fragment
__device__ __forceinline__ bf16x8 pack_acc(const f32x16& a, int half) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__bf16)a[half * 8 + e];
    return v;
}
// row index (0..31) that register r of a 32x32 accumulator holds in this lane
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }
// Kept decisions.  A hash per two decisions, 8 vector instructions each, is what a pass over the probabilities costs beyond an undropped
// one (19 where a lane's probabilities are not neighbours, as in dK/dV); the forward leaves the decisions as bits instead, for
// both backward passes, where its caller has room for them: 8 x 16 heads of 64, 1024 keys, dropout: unmasked backward 201 -> 171 us, forward
// 80 either way, causal 118 -> 109 and 47 -> 48.  A forward that keeps none is a kernel of its own: putting bits together costs an
// instruction a decision and 14 to 30 registers (with them all the same, odd sequences: 8 x 16, 1023 padded 84 us, 69 without; 2 x 12, 1021 unmasked
// 34.5, 32.9; 8 x 8 heads, 175 9.8, 9.6; 4 x 8 of 128, 501 25.4, 24.7).
// Layout: [batch, heads][queries / 32][keys / 32, tiles of 64 in full][32 words]; a word has the decisions of a query, bit j that of
// the j-th of 32 keys; the words lie in the order of accumulator rows, those of register r of the lower and the upper half wave next
// to each other: 64 bits that select lanes as they are.
__host__ __device__ __forceinline__ int64_t keep_blocks(int seq) { return (int64_t)((seq + 31) / 32) * ((seq + 63) / 64 * 2); }   // per head
__device__ __forceinline__ uint32_t* keep_at(const AttnArgs& a, int b, int head, int qs, int ks) {
    return a.keep + (((int64_t)b * a.heads + head) * keep_blocks(a.seq) + (int64_t)qs * ((a.seq + 63) / 64 * 2) + ks) * 32;
}
__device__ __forceinline__ int keep_word(int q) { return (q >> 3) * 8 + (q & 3) * 2 + ((q >> 2) & 1); }   // of the q-th of 32 queries
// bit of register r in a word shifted right by 4 * (lane >> 5): 8 * (r / 4) + r % 4
__device__ __forceinline__ float keep_bit(uint32_t shifted, int r, float v) {
    return __uint_as_float(__float_as_uint(v) & (uint32_t)__builtin_amdgcn_sbfe((int)shifted, 8 * (r >> 2) + (r & 3), 1));
}
__device__ __forceinline__ float keep_lanes(uint64_t lanes, float v) {
    float o;
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(o) : "v"(v), "s"(lanes));
    return o;
}
// Dropout over the sixteen accumulator registers of a lane whose rows acc_row(r, lane) are consecutive probability
// indices from `base` on: registers 4g .. 4g + 3 hold four neighbouring indices, i.e. two hash pairs when the first is
// even (in every lane, where the sequence length is), else parts of three (12 heads x 2043^2 forward: 58 us; 85 where the lanes
// of odd queries went another way).  Kept values are scaled, dropped ones zeroed;
// bit 8 * (r / 4) + r % 4 of what it returns is set where register r was kept.
template <bool PAIRS = false>
__device__ __forceinline__ uint32_t drop_acc_rows(const DropKey& k, uint64_t base, int lane, f32x16& v) {
    uint32_t kept = 0u;
    auto decide = [&](int r, bool keep) {
        v[r] = keep ? v[r] * k.scale : 0.f;
        kept |= keep ? 1u << (8 * (r >> 2) + (r & 3)) : 0u;
    };
    if (PAIRS || k.small) {              // the rule: fewer than 2^32 probabilities
        const uint32_t p0 = ((uint32_t)base >> 1) + 2 * (lane >> 5);   // 8 g + 4 (lane >> 5) is even
        const bool odd = !PAIRS && (base & 1) != 0;
        if (PAIRS || __builtin_amdgcn_ballot_w64(odd) == 0) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t x0 = bb_dropout_pair_bits32(k.k0, k.k1, p0 + 4 * g), x1 = bb_dropout_pair_bits32(k.k0, k.k1, p0 + 4 * g + 1);
                decide(4 * g, bb_keep_even(x0, k.thresh));
                decide(4 * g + 1, bb_keep_odd(x0, k.thresh));
                decide(4 * g + 2, bb_keep_even(x1, k.thresh));
                decide(4 * g + 3, bb_keep_odd(x1, k.thresh));
                asm("" : "+v"(kept));      // bits go in as they come: added up at the end they would wait in sixteen registers
                if (g & 1) __builtin_amdgcn_sched_barrier(0);
            }
            return kept;
        }
        // an odd sequence length: every other query's row starts inside a pair
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            uint32_t x[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) x[j] = bb_dropout_pair_bits32(k.k0, k.k1, p0 + 4 * g + j);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // the 16 bits of element e: half e % 2 of pair e / 2, or of the one further on where the first index is odd
                const uint32_t even_bits = e & 1 ? x[e >> 1] >> 16 : x[e >> 1] & 0xffffu;
                const uint32_t odd_bits = e & 1 ? x[(e + 1) >> 1] & 0xffffu : x[e >> 1] >> 16;
                decide(4 * g + e, (odd ? odd_bits : even_bits) >= k.thresh);
            }
            asm("" : "+v"(kept));
            __builtin_amdgcn_sched_barrier(0);
        }
        return kept;
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint64_t i0 = base + 8 * g + 4 * (lane >> 5);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            decide(4 * g + e, bb_dropout_keep(k.k0, k.k1, k.thresh, i0 + e));
    }
    return kept;
}

// the value of lane ^ 32
__device__ __forceinline__ float other_half(float v) {
    typedef __attribute__((ext_vector_type(2))) unsigned u2;
    const u2 w = __builtin_bit_cast(u2, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    return __uint_as_float((threadIdx.x & 32) ? w[0] : w[1]);
}
template <int N> __device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void block_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// number of leading keys a query may see (mask applied as in the reference: keep kv < limit)
__device__ __forceinline__ int kv_limit(const AttnArgs& a, int b, int q) {
    if (a.mask == BB_MASK_CAUSAL) return min(a.seq, q + 1);
    if (a.mask == BB_MASK_KEY_PADDING) return min(a.seq, a.key_len[b]);
    return a.seq;
}

// Block -> (row block, batch*head) map for a 1-D grid of 8 * ceil(nbh / 8) * nblk blocks.  The
// hardware deals consecutive block ids round-robin over the 8 XCDs, so the low three bits of
// the id pick the XCD.  Each XCD is given whole (batch, head) pairs - all their row blocks, so
// the pair's K and V stay in that XCD's L2 - and, under a causal mask, the same mix of long and
// short blocks as every other XCD, longest first (rank 0 = most work).
struct BlockMap { int rank, bh; };
__device__ __forceinline__ BlockMap map_block(int block, int nbh) {
    const int per_xcd = (nbh + 7) >> 3;
    const int xcd = block & 7, j = block >> 3;
    return {j / per_xcd, (j % per_xcd) * 8 + xcd};
}
static unsigned attn_grid(int seq, int rows, int nbh) { return (unsigned)(8 * ((nbh + 7) / 8) * ((seq + rows - 1) / rows)); }

// A block has W waves of 32 rows each, and G groups of such waves that share the walk over the tiles (group g: tiles g, g + G,
// ...; a ring each); what the groups have summed up meets in LDS at the end, added in group order.  One group of four where the
// grid gives every CU more than one block; below that what bounds a launch is a wave's walk over its tiles with nobody beside it on
// its SIMD, so the walk is shared, and where half the CUs had no block the blocks are halved too (measured: see attn_shape).
// this wave's column tiles of those the other groups have for the same rows: parts holds [group][wave][tiles][16][64] floats
template <int DW, int G, int T> __device__ __forceinline__ void attn_park(float* parts, int grp, int w, int lane, const f32x16 (&v)[T]) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) parts[(((grp * DW + w) * T + t) * 16 + r) * 64 + lane] = v[t][r];
}

enum { NODROP = 0, MADE = 1, KEPT = 2, PAIRS = 3 };

// =========================================================================================
// forward: block = 128 queries (4 waves x 32; W, G: see above), loop over 64-key tiles
// =========================================================================================
// HP: heads per block (1: one head, 2: a pair of 32-wide heads, W waves each); NPAN: 64-wide column panels of a head (1; 2 for
// 128-wide heads, HP = 1: a tile in LDS is then two [64][64] panels behind each other, each in the format above);
// DROP: no dropout; its decisions made from the key, in the forward apart from the case where all of a lane's indices go in whole pairs
// (even sequences, fewer than 2^32 probabilities; branches between the ways to make them cost moves and a wave in three); read from
// what the forward kept, in the backward
// KS k-steps of a head's scores, DT 32-wide output tiles of a head
// waves a SIMD: at least, for the registers; at most, for kernels whose LDS lets no more in (128-wide heads, four rings).  Told of three they could
// not have anyhow, the compiler read V from LDS in front of each matrix instruction, a wait each, on 160 and 115 registers; in the order of 209 and
// 132 (us): 1 x 2 heads of 128, 1150 causal 28.1 -> 25.5, 2 x 8, 2000 58.5 -> 48.7; two waves in four groups 1 x 2 of 64, 1500 causal 14.9 ->
// 14.1, 2 x 8, 1024 12.1 -> 11.7.  (Two waves in two groups: 1 x 12, 2043 causal 23.3 -> 21.5, padded 17.0 -> 17.7, 1 x 22, 2000 25.3 -> 26.8: not.)
constexpr int attn_fwd_most(int drop, int npan, int g) { return drop == NODROP && (npan == 2 || g == 4) ? 2 : 8; }
constexpr int attn_fwd_waves(int drop, int npan, int g) { return npan == 1 && g == 1 ? (drop == NODROP ? 4 : drop == PAIRS ? 3 : 2) : 2; }
template <int DROP, int HP, int NPAN = 1, int W = 4, int G = 1, bool KEEP = false>
__global__ __launch_bounds__(W * HP * G * 64) __attribute__((amdgpu_waves_per_eu(attn_fwd_waves(DROP, NPAN, G), attn_fwd_most(DROP, NPAN, G))))
void attn_fwd_kernel(const AttnArgs a) {
    static_assert(HP == 1 || NPAN == 1, "pairs of heads are 32 wide");
    constexpr int KS = 4 * NPAN / HP, DT = 2 * NPAN / HP, TILE = NPAN * 8192, ROWS = W * 32, DW = W * HP;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];  // G rings of 2 stages of K, then 2 of V
    const int tid = threadIdx.x, lane = tid & 63, uw = __builtin_amdgcn_readfirstlane(tid >> 6), dw = uw % DW, grp = G == 1 ? 0 : uw / DW;
    const int wave = dw % W, hh = HP == 1 ? 0 : dw / W;     // rows and head of the pair; of a tile's transfers, the part dw
    unsigned char* smem = smem_all + grp * (4 * TILE);
    const int groups = a.heads / HP;
    const BlockMap bm = map_block(blockIdx.x, a.batch * groups);
    if (bm.bh >= a.batch * groups) return;
    const int qb = (a.seq + ROWS - 1) / ROWS - 1 - bm.rank;  // long (late) query blocks first
    const int b = bm.bh / groups, hg = bm.bh % groups, head = hg * HP + hh;
    const int64_t row_base = (int64_t)b * a.seq;
    const bf16* Q = a.q + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* K = a.k + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* V = a.v + row_base * a.ld_qkv + hg * (64 * NPAN);
    const int q0 = qb * ROWS + wave * 32;
    const int myq = q0 + (lane & 31);
    const int last = a.seq - 1;

    // block-wide key range
    int kv_end = a.seq;
    if (a.mask == BB_MASK_CAUSAL) kv_end = min(a.seq, qb * ROWS + ROWS);
    else if (a.mask == BB_MASK_KEY_PADDING) kv_end = min(a.seq, a.key_len[b]);
    const int ntiles = (kv_end + 63) / 64, iters = (ntiles + G - 1) / G;
    const int my_limit = kv_limit(a, b, myq);
    const int wave_min_limit = kv_limit(a, b, q0);  // limits grow with the query index
    // waves whose queries all precede a tile have nothing to add (causal), nor have those past the end
    const int live_tiles = q0 >= a.seq ? 0 : a.mask == BB_MASK_CAUSAL ? min(ntiles, (q0 + 31) / 64 + 1) : ntiles;

    const LaneOff<DW> lo = lane_off<DW>(a.ld_qkv, dw, lane);
    auto issue = [&](const bf16* src, int t, unsigned char* to) {
#pragma unroll
        for (int p = 0; p < NPAN; ++p) dma_tile64<DW>(src + p * 64, a.ld_qkv, t * 64, last, to + p * 8192, dw, lane, lo);
    };
    auto issue_k = [&](int t, int slot) { if (t < ntiles) issue(K, t, smem + slot * TILE); };
    auto issue_v = [&](int t, int slot) { if (t < ntiles) issue(V, t, smem + (2 + slot) * TILE); };
    issue_k(grp, 0);
    issue_v(grp, 0);
    bf16x8 qf[KS];
    {
        const bf16* qp = Q + (int64_t)min(myq, last) * a.ld_qkv + hh * 32 + (lane >> 5) * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8*)(qp + ks * 16);
    }
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
    float m = -INFINITY, lsum = 0.f;

    auto scores = [&](const unsigned char* kt, f32x16 (&s)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const int ks = hh * 2 + k;   // k-step ks: panel ks / 4, step ks % 4 inside it
                s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_kc(kt + (ks >> 2) * 8192, u * 32, ks & 3, lane), qf[k], s[u], 0, 0, 0);
            }
        }
    };
    // masking only on tiles that reach past the first key some query of this wave may not see
    auto mask_tile = [&](int kv0, f32x16 (&s)[2]) {
        if (kv0 + 64 > wave_min_limit) {
            asm volatile("" ::: "memory");   // a real branch
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kv = kv0 + u * 32 + acc_row(r, lane);
                    s[u][r] = kv < my_limit ? s[u][r] : -INFINITY;
                }
        }
    };
    auto add_tile = [&](const unsigned char* vt, int kv0, f32x16 (&s)[2]) {
        // running max on the raw scores (the scale is positive)
        float tmax = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[u][r]);
        tmax = fmaxf(tmax, other_half(tmax)) * a.scale_log2;
        const float mnew = fmaxf(m, tmax);
        const float msafe = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __builtin_amdgcn_exp2f(m - msafe);  // m = -inf -> 0
        float psum = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = __builtin_amdgcn_exp2f(fmaf(s[u][r], a.scale_log2, -msafe));
                s[u][r] = p;
                psum += p;
            }
        lsum = lsum * alpha + psum;
        m = mnew;
        if (DROP != NODROP) asm volatile("" : "+v"(lsum));   // here: left for later, the sum keeps the probabilities beside the dropped-out ones
        if (DROP != NODROP) {   // the normaliser takes every probability, the context only the kept ones
            const uint64_t base = prob_index(a, b, head, min(myq, last)) + kv0;
            uint32_t kept[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) kept[u] = drop_acc_rows<DROP == PAIRS>(a.drop, base + u * 32, lane, s[u]);
            if constexpr (KEEP) {
                // the halves of a wave have each other's nibbles; the lower one stores the words of the first 32 keys
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    kept[u] <<= 4 * (lane >> 5);
                    kept[u] |= __float_as_uint(other_half(__uint_as_float(kept[u])));
                }
                keep_at(a, b, head, q0 / 32, kv0 / 32)[(lane >> 5) * 32 + keep_word(lane & 31)] = lane < 32 ? kept[0] : kept[1];
            }
        }
        if (__any(alpha != 1.0f)) {  // wave-uniform: once the maxima have settled nothing is rescaled
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
        }
        // O^T += V^T P^T
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const bf16x8 pf = pack_acc(s[kk >> 1], kk & 1);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const int dt = hh + d;   // output tile dt: panel dt / 2, columns (dt % 2) * 32 inside it
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_tr(vt + (dt >> 1) * 8192, kk * 16, (dt & 1) * 32, lane), pf, o[d], 0, 0, 0);
            }
        }
    };

    // The first tile and the queries: waited for in full, or the compiler, which counts its own loads only, puts the waits for the
    // queries into the loop, where they hold for the transfers of the next tile (8 x 16 heads of 64, 1024 causal 37.7 -> 34.6 us).
    asm volatile("" ::: "memory");
    wait_vm<0>();
    for (int i = 0; i < iters; ++i) {   // the barriers are the block's: every group goes round as often
        const int t = i * G + grp, slot = i & 1;
        asm volatile("" ::: "memory");
        if (t + G < ntiles) {
            issue_k(t + G, slot ^ 1);
            issue_v(t + G, slot ^ 1);
            wait_vm<16 / DW * NPAN>();
        } else {
            wait_vm<0>();
        }
        block_sync();
        if (t < live_tiles) {
            f32x16 s[2];
            scores(smem + slot * TILE, s);
            mask_tile(t * 64, s);
            add_tile(smem + (2 + slot) * TILE, t * 64, s);
        }
        block_sync();
    }
    if constexpr (G > 1) {
        // each group's context against the maximum of all of them; the first DT groups finish a column tile each
        float* stats = (float*)smem_all + DW * G * DT * 1024;   // [group][wave][m, sum][64]
        attn_park<DW, G>((float*)smem_all, grp, dw, lane, o);
        stats[((grp * DW + dw) * 2) * 64 + lane] = m;
        stats[((grp * DW + dw) * 2 + 1) * 64 + lane] = lsum;
        __syncthreads();
        float scale[G];
        float all = -INFINITY, sum = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) all = fmaxf(all, stats[((g * DW + dw) * 2) * 64 + lane]);
        const float safe = all == -INFINITY ? 0.f : all;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            scale[g] = __builtin_amdgcn_exp2f(stats[((g * DW + dw) * 2) * 64 + lane] - safe);
            sum += stats[((g * DW + dw) * 2 + 1) * 64 + lane] * scale[g];
        }
        m = all;
        lsum = sum;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            if (dt % G != grp) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float v = 0.f;
#pragma unroll
                for (int g = 0; g < G; ++g) v += ((float*)smem_all)[(((g * DW + dw) * DT + dt) * 16 + r) * 64 + lane] * scale[g];
                o[dt][r] = v;
            }
        }
    }
    lsum += other_half(lsum);
    const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
    if (myq < a.seq) {
        bf16* op = a.out + (row_base + myq) * a.ld_o + hg * (64 * NPAN) + hh * 32;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            if (dt % G != grp) continue;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d = dt * 32 + 8 * g4 + 4 * (lane >> 5);
                u32x2 w = {pack2bf(o[dt][g4 * 4] * inv, o[dt][g4 * 4 + 1] * inv),
                           pack2bf(o[dt][g4 * 4 + 2] * inv, o[dt][g4 * 4 + 3] * inv)};
                *(u32x2*)(op + d) = w;
            }
        }
        if (lane < 32 && grp == 0) a.lse[((int64_t)b * a.heads + head) * a.seq + myq] = m + log2f(lsum);
    }
}

// =========================================================================================
// backward: the walk of a wave over its sub-tiles, shared by both kernels
// =========================================================================================
// A sub-tile's work is a chain: scores (matrix cores, operands from LDS), probabilities (vector ALU) with the gradients of the scores
// beside them (matrix cores), dS (vector ALU), the products with P and dS (matrix cores).  PIPE: the scores of the sub-tile after it
// go beside dS, so that a wave starts a sub-tile on the vector ALU at once, and operands are read from LDS a phase ahead.  What it gives
// is latency, where a SIMD has one wave: 2 x 8 heads of 64, 1024 keys 38.2 us one after the other, 33.1 this way.  Beyond that the two are
// equal (8 x 16 heads, 1024: 140 us, 865 TFLOP/s of matrix work; two, three or four waves a SIMD the same within 3 %; without the
// exponentials 121, without LDS reads 118): no one of them bounds it, and neither does power alone (causal, of a CU in use: matrix
// pipe 33 %, vector ALU 35 to 45 %, at 2.2 to 2.3 of 2.4 GHz).  A wave walks only sub-tiles of 32 that
// hold a pair its mask keeps; with the waits outside of the loop (below) 8 x 16 heads, 1024 causal 100.8 -> 90.9, unmasked 157 -> 139.
constexpr bool attn_bwd_pipe(int npan) { return npan == 1; }
// stages of a ring: three where a tile's last products come behind the barrier that hands the next tile out, two where three do not fit
constexpr int attn_bwd_stages(int npan, int g) { return npan == 1 && g <= 2 ? 3 : 2; }
template <int G, int STAGES, int STAGE, bool PIPE, typename Live, typename FetchS, typename FetchG, typename Scores, typename Grads,
          typename Probs, typename Contract, typename Issue>
__device__ __forceinline__ void attn_bwd_walk(unsigned char* smem, int t, int iters, const Live& live, const FetchS& fetch_scores,
                                              const FetchG& fetch_grads, const Scores& scores, const Grads& score_grads,
                                              const Probs& probs, const Contract& contract, const Issue& issue) {
    using First = std::integral_constant<int, 0>;
    int stage = 0;
    auto begin = [&](const unsigned char* st, auto j_c) {      // a wave's first sub-tile, or the first behind a turn it could not look past
        fetch_scores(st, j_c);
        fetch_grads(st, j_c);
        scores(j_c);
    };
    if constexpr (PIPE) {
        if (live(t, 0)) begin(smem, First{});
    }
    for (int i = 0; i < iters; ++i, t += G) {   // the barriers are the block's: every group goes round as often
        const unsigned char* st = smem + stage * STAGE;
        const int after = stage + 1 == STAGES ? 0 : stage + 1, free = STAGES == 2 ? stage : after + 1 == STAGES ? 0 : after + 1;
        const unsigned char* st_after = smem + after * STAGE;
        // the next tile, on its way for a whole tile by now, has landed for all waves; all are done with the stage that the one
        // after it is sent to
        auto turn = [&]() {
            if (i + 1 < iters) {
                asm volatile("" ::: "memory");
                wait_vm<0>();
                block_sync();
                issue(t + 2 * G, free);
            }
        };
        auto step = [&](auto j_c) {
            constexpr int j = decltype(j_c)::value;
            constexpr bool LAST = j == 1;
            constexpr bool BEHIND = LAST && STAGES == 2;      // the next tile comes in behind the last products of this one
            using Next = std::integral_constant<int, LAST ? 0 : j + 1>;
            const bool run = live(t, j), next = LAST ? i + 1 < iters && live(t + G, 0) : live(t, j + 1);
            if constexpr (PIPE && LAST && STAGES == 3) turn();
            const unsigned char* st_next = LAST ? st_after : st;
            if (run) {
                if constexpr (!PIPE) begin(st, j_c);
                // (of no use behind the wave's last sub-tile: branches around them would keep them apart from what they go beside)
                if constexpr (PIPE && !BEHIND) fetch_scores(st_next, Next{});
                score_grads(j_c);
                probs(st, t, j_c);
                if constexpr (PIPE && !BEHIND) {
                    fetch_grads(st_next, Next{});
                    scores(Next{});
                }
                contract(st, t, j_c);
            } else if constexpr (PIPE && !BEHIND) {
                if (next) begin(st_next, Next{});
            }
            if constexpr (LAST && STAGES == 2) {
                turn();
                if (PIPE && next) begin(st_after, Next{});
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        stage = after;
    }
}

// =========================================================================================
// backward dK, dV: block = 128 keys (4 waves x 32), loop over 64-query tiles
// =========================================================================================
// NPAN = 2 (128-wide heads): a block accumulates dK and dV for ONE 64-wide half `fh` of the head's columns (the grid
// has two blocks per head and key block); scores and dP take the full 128 columns in both, i.e. are made twice -- a wave
// that held all four output tiles of dK and of dV next to K, V, S and dP would need more registers than it has.
// OWN: no dQ kernel has run before this one: the block makes delta of all its queries itself, in LDS from OWN_AT on
template <int DROP, int HP, int NPAN, int W, int G, bool OWN>
__device__ __forceinline__ void attn_bwd_dkv_block(const AttnArgs& a, const int block, unsigned char* smem_all, const int own_at) {
    static_assert(HP == 1 || NPAN == 1, "pairs of heads are 32 wide");
    constexpr int KS = 4 * NPAN / HP, DT = 2 / HP, TILE = NPAN * 8192, ROWS = W * 32, DW = W * HP;
    // per group STAGES x (Q tile, dO tile: 8 KiB per panel, lse 256 B per head, delta 256 B per head)
    constexpr bool PIPE = attn_bwd_pipe(NPAN);
    constexpr int STAGE = 2 * TILE + 512 * HP, STAGES = attn_bwd_stages(NPAN, G), BUFS = PIPE ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, uw = __builtin_amdgcn_readfirstlane(tid >> 6), dw = uw % DW, grp = G == 1 ? 0 : uw / DW;
    const int wave = dw % W, hh = HP == 1 ? 0 : dw / W;
    unsigned char* smem = smem_all + grp * (STAGES * STAGE);
    const int groups = a.heads / HP;
    const BlockMap bm = map_block(block, a.batch * groups * NPAN);
    if (bm.bh >= a.batch * groups * NPAN) return;
    const int kb = bm.rank;  // early key blocks are seen by the most queries
    const int fh = bm.bh % NPAN, bg = bm.bh / NPAN;
    const int b = bg / groups, hg = bg % groups, head0 = hg * HP, head = head0 + hh;
    const int64_t row_base = (int64_t)b * a.seq;
    const bf16* Q = a.q + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* K = a.k + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* V = a.v + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* DO = a.d_o + row_base * a.ld_o + hg * (64 * NPAN);
    // the statistics of the block's heads lie behind each other: [batch, heads, seq]
    const float* LSE = a.lse + ((int64_t)b * a.heads + head0) * a.seq;
    const float* DELTA = a.delta + ((int64_t)b * a.heads + head0) * a.seq;
    const int kv0 = kb * ROWS + wave * 32;
    const int mykv = kv0 + (lane & 31);
    const int last = a.seq - 1;
    const int pad_limit = a.mask == BB_MASK_KEY_PADDING ? min(a.seq, a.key_len[b]) : a.seq;

    // query range that can see keys of this block
    const int q_begin = a.mask == BB_MASK_CAUSAL ? (kb * ROWS) / 64 : 0;  // first 64-query tile
    // a block whose keys are all padding has nothing to accumulate: it only stores its zeros
    const int ntiles = kb * ROWS >= pad_limit ? 0 : (a.seq + 63) / 64;

    const LaneOff<DW> lo = lane_off<DW>(a.ld_qkv, dw, lane), lo_o = lane_off<DW>(a.ld_o, dw, lane);
    auto issue = [&](int t, int slot) {
        unsigned char* st = smem + slot * STAGE;
        const int qs = t * 64;
#pragma unroll
        for (int p = 0; p < NPAN; ++p) {
            dma_tile64<DW>(Q + p * 64, a.ld_qkv, qs, last, st + p * 8192, dw, lane, lo);
            dma_tile64<DW>(DO + p * 64, a.ld_o, qs, last, st + TILE + p * 8192, dw, lane, lo_o);
        }
        // extra loads, dealt to the waves: lse of the block's heads, then delta
#pragma unroll
        for (int j = 0; j < (OWN ? 1 : 2) * HP; ++j)
            if (j % DW == dw) dma_f32x64((j / HP ? DELTA : LSE) + (int64_t)(j % HP) * a.seq, qs, last, st + 2 * TILE + j * 256, lane);
    };
    const int t0 = q_begin + grp, iters = max(0, (ntiles - q_begin + G - 1) / G);
    if (t0 < ntiles) issue(t0, 0);
    if (t0 + G < ntiles) issue(t0 + G, 1);
    bf16x8 kf[KS], vf[KS];
    {
        const int64_t off = (int64_t)min(mykv, last) * a.ld_qkv + hh * 32 + (lane >> 5) * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            kf[ks] = *(const bf16x8*)(K + off + ks * 16);
            vf[ks] = *(const bf16x8*)(V + off + ks * 16);
        }
    }
    f32x16 dk[DT], dv[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) dk[t][r] = dv[t][r] = 0.f;

    const int own_rows = (a.seq + 63) / 64 * 64;     // of a head's deltas in LDS
    if constexpr (OWN) {
        // as the dQ kernel makes them, in its order of additions: a lane and its partner (lane ^ 32) have the halves of each
        // 16-column step of a row
        float* own = (float*)(smem_all + own_at);
        const bf16* O = a.o + row_base * a.ld_o + hg * (64 * NPAN);
        for (int q = q_begin * 64 + (tid >> 6) * 32 + (lane & 31); q < ntiles * 64; q += DW * G * 32) {
            const int64_t at = (int64_t)min(q, last) * a.ld_o + (lane >> 5) * 8;
            bf16x8 df[4 * NPAN], of[4 * NPAN];
#pragma unroll
            for (int ks = 0; ks < 4 * NPAN; ++ks) {
                df[ks] = *(const bf16x8*)(DO + at + ks * 16);
                of[ks] = *(const bf16x8*)(O + at + ks * 16);
            }
#pragma unroll
            for (int hd = 0; hd < HP; ++hd) {
                float dl = 0.f;
#pragma unroll
                for (int k = 0; k < KS; ++k)
#pragma unroll
                    for (int e = 0; e < 8; ++e) dl = fmaf((float)df[hd * KS + k][e], (float)of[hd * KS + k][e], dl);
                dl += other_half(dl);
                if (lane < 32) own[hd * own_rows + q] = dl;
            }
        }
        // (the first tile's wait and barrier make them visible)
    }
    // the wave's sub-tiles of 32 queries: not those that all precede its keys, nor any for keys past the end or all padding
    const int sub_begin = a.mask == BB_MASK_CAUSAL ? kv0 / 32 : 0, sub_end = kv0 >= pad_limit ? 0 : (a.seq + 31) / 32;
    auto live = [&](int t, int u) { const int sub = t * 2 + u; return t < ntiles && sub >= sub_begin && sub < sub_end; };
    f32x16 s[BUFS], dp;
    // operands of the scores S and of their gradients dP, from LDS
    bf16x8 fs[KS], fdp[KS];
    auto fetch_scores = [&](const unsigned char* st, auto j_c) {
        constexpr int u = decltype(j_c)::value;
#pragma unroll
        for (int k = 0; k < KS; ++k) fs[k] = frag_kc(st + ((hh * 2 + k) >> 2) * 8192, u * 32, (hh * 2 + k) & 3, lane);
    };
    auto fetch_grads = [&](const unsigned char* st, auto j_c) {
        constexpr int u = decltype(j_c)::value;
#pragma unroll
        for (int k = 0; k < KS; ++k) fdp[k] = frag_kc(st + TILE + ((hh * 2 + k) >> 2) * 8192, u * 32, (hh * 2 + k) & 3, lane);
    };
    auto scores = [&](auto j_c) {
        constexpr int n = decltype(j_c)::value % BUFS;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k) s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fs[k], kf[k], s[n], 0, 0, 0);
    };
    auto score_grads = [&](auto j_c) {
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k) dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fdp[k], vf[k], dp, 0, 0, 0);
    };
    // P = exp2(S * c - lse[q]); rows q = acc_row(r), column kv = lane.  Only sub-tiles on the causal diagonal or past the last query
    // mask per element; keys beyond the padding limit are whole lanes and are cleared once, after the loop.
    typedef __attribute__((ext_vector_type(8))) uint64_t u64x8;
    u64x8 lanes[2];     // kept decisions of the sub-tile: register r's lanes
    auto probs = [&](const unsigned char* st, int t, auto j_c) {
        constexpr int u = decltype(j_c)::value, n = u % BUFS;
        if (DROP == KEPT) {
            const auto* w = (const __attribute__((address_space(4))) u64x8*)(uintptr_t)keep_at(a, b, head, t * 2 + u, kv0 / 32);
            lanes[0] = w[0];
            lanes[1] = w[1];
        }
        const float* lse_t = (const float*)(st + 2 * TILE) + 64 * hh;
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const int ql = u * 32 + 8 * g4 + 4 * (lane >> 5);
            const f32x4 l4 = *(const f32x4*)(lse_t + ql);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[n][g4 * 4 + e] = __builtin_amdgcn_exp2f(fmaf(s[n][g4 * 4 + e], a.scale_log2, -l4[e]));
        }
        const int qs = t * 64 + u * 32;
        if ((a.mask == BB_MASK_CAUSAL && qs < kv0 + 31) || qs + 32 > a.seq) {
            asm volatile("" ::: "memory");  // a real branch: most sub-tiles skip it
            const int qlane = qs + 4 * (lane >> 5);  // register r holds query qlane + 8*(r/4) + r%4
            const int qmin = a.mask == BB_MASK_CAUSAL ? mykv : 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int q = qlane + 8 * (r >> 2) + (r & 3);
                s[n][r] = q >= qmin && q < a.seq ? s[n][r] : 0.f;
            }
        }
    };
    // dS = P * (dP - delta[q]), then dV^T += dO^T P~ ; dK^T += Q^T dS (contraction over the 32 queries of the sub-tile)
    auto contract = [&](const unsigned char* st, int t, auto j_c) {
        constexpr int u = decltype(j_c)::value, n = u % BUFS;
        const float* del_t = OWN ? (const float*)(smem_all + own_at) + hh * own_rows + t * 64 : (const float*)(st + 2 * TILE) + 64 * HP + 64 * hh;
        // dropout: dP = dP~ o mask / (1 - p) before it meets P; P itself is masked (into what multiplied V in
        // the forward) only after dS has been formed from the unmasked probabilities
        unsigned kept = 0u;   // bit r (sixteen booleans cost the registers that K, V and the sums leave)
        if (DROP == KEPT) {
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = keep_lanes(lanes[r >> 3][r & 7], dp[r] * a.drop.scale);
        } else if (DROP == MADE) {
            asm volatile("" ::: "memory");
            const int qlane = t * 64 + u * 32 + 4 * (lane >> 5);
            if (a.drop.small) {
                // 32-bit indices; what is decided for a query past the end (masked out above) or a key past it (a whole
                // lane, never stored) does not matter
                const uint32_t i0 = ((uint32_t)(b * a.heads + head) * (uint32_t)a.seq + (uint32_t)qlane) * (uint32_t)a.seq + (uint32_t)mykv;
                if (a.seq % 2 == 0) {
                    // Rows start even: lanes 2j and 2j + 1 (keys 2j, 2j + 1) need the two halves of one hash in every row.
                    // Of two rows the even lane hashes the first and the odd lane the second, and they exchange the
                    // other's halves: a hash (two quarter-rate multiplies) per two decisions, as where the indices of a
                    // lane are neighbours.  (Backward of 8 x 16 heads x 1024^2 probabilities: 238 us with a hash per decision,
                    // 223 with this; 128-wide heads, 2 x 8 x 512^2 causal: 89 and 67.)
                    const uint32_t own = (lane & 1) * 16, other = 16 - own;
                    const uint32_t j0 = i0 + (lane & 1) * (uint32_t)a.seq;
                    uint32_t km = 0u, kt = 0u;   // bit r: this lane's decision of its row, the neighbour's row
#pragma unroll
                    for (int r = 0; r < 16; r += 2) {
                        const uint32_t at = j0 + (uint32_t)(8 * (r >> 2) + (r & 3)) * (uint32_t)a.seq;
                        const uint32_t x = bb_dropout_pair_bits32(a.drop.k0, a.drop.k1, at >> 1);
                        const bool mine = ((x >> own) & 0xffffu) >= a.drop.thresh;
                        const uint32_t sent =
                            (uint32_t)__builtin_amdgcn_mov_dpp((int)((x >> other) & 0xffffu), 0xb1 /* quad_perm 1 0 3 2 */, 0xf, 0xf, true);
                        const bool theirs = sent >= a.drop.thresh;
                        km |= mine ? 1u << r : 0u;
                        kt |= theirs ? 1u << r : 0u;
                    }
                    kept = (lane & 1) ? km << 1 | kt : km | kt << 1;
                } else {
#pragma unroll 2                        // (unrolled whole, this and the next loop cost the first one's registers)
                    for (int r = 0; r < 16; ++r) {
                        const uint32_t idx = i0 + (uint32_t)(8 * (r >> 2) + (r & 3)) * (uint32_t)a.seq;
                        const uint32_t x = bb_dropout_pair_bits32(a.drop.k0, a.drop.k1, idx >> 1);
                        kept |= (((x >> ((idx & 1) * 16)) & 0xffffu) >= a.drop.thresh ? 1u : 0u) << r;
                    }
                }
            } else {
#pragma unroll 1
                for (int r = 0; r < 16; ++r) {
                    const int q = min(qlane + 8 * (r >> 2) + (r & 3), last);
                    kept |= (bb_dropout_keep(a.drop.k0, a.drop.k1, a.drop.thresh, prob_index(a, b, head, q) + min(mykv, last)) ? 1u : 0u) << r;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = (kept >> r) & 1u ? dp[r] * a.drop.scale : 0.f;
        }
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const int ql = u * 32 + 8 * g4 + 4 * (lane >> 5);
            const f32x4 d4 = *(const f32x4*)(del_t + ql);
#pragma unroll
            for (int e = 0; e < 4; ++e) dp[g4 * 4 + e] = s[n][g4 * 4 + e] * (dp[g4 * 4 + e] - d4[e]);
        }
        if (DROP == KEPT) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = keep_lanes(lanes[r >> 3][r & 7], s[n][r] * a.drop.scale);
        } else if (DROP == MADE) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = (kept >> r) & 1u ? s[n][r] * a.drop.scale : 0.f;
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            if (PIPE && kk) __builtin_amdgcn_sched_barrier(0);   // (the fragments of both halves at once find no registers)
            const bf16x8 pf = pack_acc(s[n], kk), dsf = pack_acc(dp, kk);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const int col = (hh + d) * 32;
                dv[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_tr(st + TILE + fh * 8192, u * 32 + kk * 16, col, lane), pf, dv[d], 0, 0, 0);
                dk[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag_tr(st + fh * 8192, u * 32 + kk * 16, col, lane), dsf, dk[d], 0, 0, 0);
            }
        }
    };
    if (iters > 0) {
        asm volatile("" ::: "memory");
        wait_vm<0>();      // in full: a wait the compiler left for its own loads would stand in the loop, in front of every transfer
        block_sync();
        attn_bwd_walk<G, STAGES, STAGE, PIPE>(smem, t0, iters, live, fetch_scores, fetch_grads, scores, score_grads, probs, contract,
                                              [&](int t, int slot) { if (t < ntiles) issue(t, slot); });
        if constexpr (G > 1) block_sync();     // the rings are done with
    }
    if constexpr (G > 1) {
        // the groups' sums, first dV, then dK (one after the other: together they would not find room)
        float* parts = (float*)smem_all;
        auto join = [&](f32x16 (&v)[DT]) {
            attn_park<DW, G>(parts, grp, dw, lane, v);
            __syncthreads();
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                if (t % G != grp) continue;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float x = parts[((dw * DT + t) * 16 + r) * 64 + lane];
#pragma unroll
                    for (int g = 1; g < G; ++g) x += parts[(((g * DW + dw) * DT + t) * 16 + r) * 64 + lane];
                    v[t][r] = x;
                }
            }
            __syncthreads();
        };
        join(dv);
        join(dk);
    }
    if (mykv >= pad_limit) {  // a padded key takes no probability mass: its gradients are zero
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) dk[t][r] = dv[t][r] = 0.f;
    }
    if (mykv < a.seq) {
        bf16* dkp = a.dk + (row_base + mykv) * a.ld_dqkv + hg * (64 * NPAN) + fh * 64 + hh * 32;
        bf16* dvp = a.dv + (row_base + mykv) * a.ld_dqkv + hg * (64 * NPAN) + fh * 64 + hh * 32;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                if (dt % G != grp) continue;
                const int d = dt * 32 + 8 * g4 + 4 * (lane >> 5);
                u32x2 wk = {pack2bf(dk[dt][g4 * 4] * a.scale, dk[dt][g4 * 4 + 1] * a.scale),
                            pack2bf(dk[dt][g4 * 4 + 2] * a.scale, dk[dt][g4 * 4 + 3] * a.scale)};
                u32x2 wv = {pack2bf(dv[dt][g4 * 4], dv[dt][g4 * 4 + 1]), pack2bf(dv[dt][g4 * 4 + 2], dv[dt][g4 * 4 + 3])};
                *(u32x2*)(dkp + d) = wk;
                *(u32x2*)(dvp + d) = wv;
            }
    }
}

// =========================================================================================
// backward dQ: block = 128 queries (4 waves x 32), loop over 64-key tiles
// =========================================================================================
// OWN: the dK / dV blocks of the launch make their deltas themselves, nobody reads this block's
template <int DROP, int HP, int NPAN, int W, int G, bool OWN>
__device__ __forceinline__ void attn_bwd_dq_block(const AttnArgs& a, const int block, unsigned char* smem_all) {
    static_assert(HP == 1 || NPAN == 1, "pairs of heads are 32 wide");
    constexpr int KS = 4 * NPAN / HP, DT = 2 * NPAN / HP, TILE = NPAN * 8192, ROWS = W * 32, DW = W * HP;
    constexpr bool PIPE = attn_bwd_pipe(NPAN);
    constexpr int STAGES = attn_bwd_stages(NPAN, G), BUFS = PIPE ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, uw = __builtin_amdgcn_readfirstlane(tid >> 6), dw = uw % DW, grp = G == 1 ? 0 : uw / DW;
    const int wave = dw % W, hh = HP == 1 ? 0 : dw / W;
    constexpr int STAGE = 2 * TILE + (DROP == KEPT ? DW * 256 : 0);      // K tile, V tile, the kept decisions of each wave's queries
    unsigned char* smem = smem_all + grp * (STAGES * STAGE);
    const int groups = a.heads / HP;
    const BlockMap bm = map_block(block, a.batch * groups);
    if (bm.bh >= a.batch * groups) return;
    const int qb = (a.seq + ROWS - 1) / ROWS - 1 - bm.rank;
    const int b = bm.bh / groups, hg = bm.bh % groups, head0 = hg * HP, head = head0 + hh;
    const int64_t row_base = (int64_t)b * a.seq;
    const bf16* Q = a.q + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* K = a.k + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* V = a.v + row_base * a.ld_qkv + hg * (64 * NPAN);
    const bf16* DO = a.d_o + row_base * a.ld_o + hg * (64 * NPAN);
    const int q0 = qb * ROWS + wave * 32;
    const int myq = q0 + (lane & 31);
    const int last = a.seq - 1;
    int kv_end = a.seq;
    if (a.mask == BB_MASK_CAUSAL) kv_end = min(a.seq, qb * ROWS + ROWS);
    else if (a.mask == BB_MASK_KEY_PADDING) kv_end = min(a.seq, a.key_len[b]);
    const int ntiles = (kv_end + 63) / 64;
    // rows past the end compute on clamped inputs and are not stored
    const int my_limit = kv_limit(a, b, myq);
    const int wave_min_limit = kv_limit(a, b, q0);  // limits grow with the query index

    const LaneOff<DW> lo = lane_off<DW>(a.ld_qkv, dw, lane);
    auto issue = [&](int t, int slot) {
        unsigned char* st = smem + slot * STAGE;
        const int kv0 = t * 64;
        if (DROP == KEPT) dma4(keep_at(a, b, head, min(q0, last) / 32, t * 2) + lane, st + 2 * TILE + dw * 256);
#pragma unroll
        for (int p = 0; p < NPAN; ++p) {
            dma_tile64<DW>(K + p * 64, a.ld_qkv, kv0, last, st + p * 8192, dw, lane, lo);
            dma_tile64<DW>(V + p * 64, a.ld_qkv, kv0, last, st + TILE + p * 8192, dw, lane, lo);
        }
    };
    if (grp < ntiles) issue(grp, 0);
    if (grp + G < ntiles) issue(grp + G, 1);
    bf16x8 qf[KS], dof[KS];
    {
        const int64_t r = min(myq, last);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            qf[ks] = *(const bf16x8*)(Q + r * a.ld_qkv + hh * 32 + (lane >> 5) * 8 + ks * 16);
            dof[ks] = *(const bf16x8*)(DO + r * a.ld_o + hh * 32 + (lane >> 5) * 8 + ks * 16);
        }
    }
    // delta[q] = rowsum(dO o O) over the head's columns: the lane and its partner (lane ^ 32) hold the two halves of
    // each 16-column step of the query's dO row; the matching halves of O are fetched once.  Written out for a
    // dK / dV kernel that runs after this one.
    float my_lse, my_delta = 0.f;
    {
        const bf16* O = a.o + row_base * a.ld_o + hg * (64 * NPAN) + hh * 32;
        const int64_t r = min(myq, last), stat = ((int64_t)b * a.heads + head) * a.seq + r;
        my_lse = a.lse[stat];
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const bf16x8 of = *(const bf16x8*)(O + r * a.ld_o + (lane >> 5) * 8 + k * 16);
#pragma unroll
            for (int e = 0; e < 8; ++e) my_delta = fmaf((float)dof[k][e], (float)of[e], my_delta);
        }
        my_delta += other_half(my_delta);
        if (!OWN && lane < 32 && myq < a.seq && grp == 0) a.delta[stat] = my_delta;
    }
    f32x16 dq[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[t][r] = 0.f;

    // the wave's sub-tiles of 32 keys: up to the last one that some query of it may see, none for queries past the end
    const int sub_end = q0 >= a.seq ? 0 : a.mask == BB_MASK_CAUSAL ? q0 / 32 + 1 : (kv_end + 31) / 32;
    auto live = [&](int t, int u) { return t < ntiles && t * 2 + u < sub_end; };
    f32x16 s[BUFS], dp;
    // operands of the scores S and of their gradients dP, from LDS
    bf16x8 fs[KS], fdp[KS];
    auto fetch_scores = [&](const unsigned char* st, auto j_c) {
        constexpr int u = decltype(j_c)::value;
#pragma unroll
        for (int k = 0; k < KS; ++k) fs[k] = frag_kc(st + ((hh * 2 + k) >> 2) * 8192, u * 32, (hh * 2 + k) & 3, lane);
    };
    auto fetch_grads = [&](const unsigned char* st, auto j_c) {
        constexpr int u = decltype(j_c)::value;
#pragma unroll
        for (int k = 0; k < KS; ++k) fdp[k] = frag_kc(st + TILE + ((hh * 2 + k) >> 2) * 8192, u * 32, (hh * 2 + k) & 3, lane);
    };
    auto scores = [&](auto j_c) {
        constexpr int n = decltype(j_c)::value % BUFS;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k) s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fs[k], qf[k], s[n], 0, 0, 0);
    };
    auto score_grads = [&](auto j_c) {
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k) dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fdp[k], dof[k], dp, 0, 0, 0);
    };
    auto probs = [&](const unsigned char*, int t, auto j_c) {
        constexpr int u = decltype(j_c)::value, n = u % BUFS;
        const int kv = t * 64 + u * 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[n][r] = __builtin_amdgcn_exp2f(fmaf(s[n][r], a.scale_log2, -my_lse));
        if (kv + 32 > wave_min_limit) {
            asm volatile("" ::: "memory");  // a real branch: only tiles on the mask boundary pay for it
            const int lim = my_limit - kv - 4 * (lane >> 5);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[n][r] = 8 * (r >> 2) + (r & 3) < lim ? s[n][r] : 0.f;
        }
    };
    auto contract = [&](const unsigned char* st, int t, auto j_c) {
        constexpr int u = decltype(j_c)::value, n = u % BUFS;
        if constexpr (DROP != NODROP) {
            asm volatile("" ::: "memory");
            if constexpr (DROP == KEPT) {
                const uint32_t w = ((const uint32_t*)(st + 2 * TILE))[dw * 64 + u * 32 + keep_word(lane & 31)] >> (4 * (lane >> 5));
#pragma unroll
                for (int r = 0; r < 16; ++r) dp[r] = keep_bit(w, r, dp[r] * a.drop.scale);
            } else {
                drop_acc_rows(a.drop, prob_index(a, b, head, min(myq, last)) + t * 64 + u * 32, lane, dp);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = s[n][r] * (dp[r] - my_delta);
        // dQ^T += K^T dS^T (contraction over the 32 keys of this sub-tile)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const bf16x8 dsf = pack_acc(dp, kk);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const int dt = hh + d;
                const bf16x8 kt = frag_tr(st + (dt >> 1) * 8192, u * 32 + kk * 16, (dt & 1) * 32, lane);
                dq[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, dsf, dq[d], 0, 0, 0);
            }
        }
    };
    const int iters = (ntiles + G - 1) / G;
    if (iters > 0) {
        asm volatile("" ::: "memory");
        wait_vm<0>();      // in full: a wait the compiler left for its own loads would stand in the loop, in front of every transfer
        block_sync();
        attn_bwd_walk<G, STAGES, STAGE, PIPE>(smem, grp, iters, live, fetch_scores, fetch_grads, scores, score_grads, probs, contract,
                                              [&](int t, int slot) { if (t < ntiles) issue(t, slot); });
        if constexpr (G > 1) block_sync();     // the rings are done with
    }
    if constexpr (G > 1) {
        float* parts = (float*)smem_all;
        attn_park<DW, G>(parts, grp, dw, lane, dq);
        __syncthreads();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            if (dt % G != grp) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float x = parts[((dw * DT + dt) * 16 + r) * 64 + lane];
#pragma unroll
                for (int g = 1; g < G; ++g) x += parts[(((g * DW + dw) * DT + dt) * 16 + r) * 64 + lane];
                dq[dt][r] = x;
            }
        }
    }
    if (myq < a.seq) {
        bf16* dqp = a.dq + (row_base + myq) * a.ld_dqkv + hg * (64 * NPAN) + hh * 32;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                if (dt % G != grp) continue;
                const int d = dt * 32 + 8 * g4 + 4 * (lane >> 5);
                u32x2 w = {pack2bf(dq[dt][g4 * 4] * a.scale, dq[dt][g4 * 4 + 1] * a.scale),
                           pack2bf(dq[dt][g4 * 4 + 2] * a.scale, dq[dt][g4 * 4 + 3] * a.scale)};
                *(u32x2*)(dqp + d) = w;
            }
    }
}

template <int DROP, int HP, int NPAN = 1, int W = 4, int G = 1>
__global__ __launch_bounds__(W * HP * G * 64, 2) void attn_bwd_dkv_kernel(const AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];
    attn_bwd_dkv_block<DROP, HP, NPAN, W, G, false>(a, blockIdx.x, smem_all, 0);
}
template <int DROP, int HP, int NPAN = 1, int W = 4, int G = 1>
__global__ __launch_bounds__(W * HP * G * 64, 2) void attn_bwd_dq_kernel(const AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];
    attn_bwd_dq_block<DROP, HP, NPAN, W, G, false>(a, blockIdx.x, smem_all);
}
// Both in one launch, where there is room for all their blocks (attn_bwd_launch): first the dK / dV blocks, whose walks are the
// longer ones, then the dQ blocks.
template <int DROP, int HP, int NPAN = 1, int W = 4, int G = 1>
__global__ __launch_bounds__(W * HP * G * 64, 2) void attn_bwd_kernel(const AttnArgs a, const int dkv_blocks, const int own_at) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];
    if ((int)blockIdx.x < dkv_blocks) attn_bwd_dkv_block<DROP, HP, NPAN, W, G, true>(a, blockIdx.x, smem_all, own_at);
    else attn_bwd_dq_block<DROP, HP, NPAN, W, G, true>(a, blockIdx.x - dkv_blocks, smem_all);
}

// =========================================================================================
// host entry points
// =========================================================================================
static int check_attn(const char* name, int dtype, int mask, int batch, int heads, int seq, int head_dim, int64_t ld_qkv,
                      int64_t ld_o, const int32_t* key_len) {
    BB_REQUIRE(dtype == BB_BF16, "%s: the fused attention kernels are bf16 only (got dtype %d)", name, dtype);
    BB_REQUIRE(head_dim == 64 || head_dim == 128 || (head_dim == 32 && heads % 2 == 0),
               "%s: head dimension must be 64, 128, or 32 with an even number of heads (got %d, %d heads)", name, head_dim, heads);
    BB_REQUIRE(mask >= BB_MASK_NONE && mask <= BB_MASK_KEY_PADDING, "%s: bad mask %d", name, mask);
    BB_REQUIRE(mask != BB_MASK_KEY_PADDING || key_len, "%s: key_padding mask needs key_len", name);
    BB_REQUIRE(batch >= 0 && heads > 0 && seq >= 0, "%s: bad shape", name);
    BB_REQUIRE(ld_qkv % 8 == 0 && ld_o % 8 == 0 && ld_qkv >= heads * head_dim && ld_o >= heads * head_dim, "%s: bad leading dimension", name);
    BB_REQUIRE(ld_qkv < (1 << 24) && ld_o < (1 << 24), "%s: leading dimension too large", name);
    BB_REQUIRE(((int64_t)batch * heads * 2 + 8) * ((seq + 127) / 128) < (1ll << 31), "%s: batch * heads * seq exceeds the grid limit", name);
    return BB_OK;
}

// LDS: the rings, or what the groups leave for each other
template <int HP, int NPAN, int W, int G> constexpr size_t attn_lds(bool bwd, bool dkv) {
    const size_t ring = G * (size_t)(bwd ? attn_bwd_stages(NPAN, G) : 2) * (2 * NPAN * 8192 + (dkv ? 512 * HP : bwd ? W * HP * 256 : 0));
    const size_t parts = G == 1 ? 0 : (size_t)W * HP * G * ((dkv ? 2 : 2 * NPAN) / HP * 4096 + (bwd ? 0 : 512));
    return ring > parts ? ring : parts;
}
template <typename K> static int attn_go(K kern, int seq, int rows, int nbh, int threads, size_t lds, const AttnArgs& a, hipStream_t st) {
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, lds));
    bb_launch(kern, dim3(attn_grid(seq, rows, nbh)), dim3(threads), lds, st, a);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
// dropout is a kernel of its own: its keep decisions cost registers that decide how many blocks a CU holds
struct attn_fwd_launch {
    template <int HP, int NPAN, int W, int G> static int go(int seq, int nbh, const AttnArgs& a, hipStream_t st) {
        const bool pairs = a.drop.small && seq % 2 == 0;
        auto kern = !a.drop.thresh ? attn_fwd_kernel<NODROP, HP, NPAN, W, G>
                    : a.keep       ? (pairs ? attn_fwd_kernel<PAIRS, HP, NPAN, W, G, true> : attn_fwd_kernel<MADE, HP, NPAN, W, G, true>)
                                   : (pairs ? attn_fwd_kernel<PAIRS, HP, NPAN, W, G> : attn_fwd_kernel<MADE, HP, NPAN, W, G>);
        return attn_go(kern, seq, W * 32, nbh, W * HP * G * 64, attn_lds<HP, NPAN, W, G>(false, false), a, st);
    }
};
struct attn_dq_launch {
    template <int HP, int NPAN, int W, int G> static int go(int seq, int nbh, const AttnArgs& a, hipStream_t st) {
        auto kern = a.keep ? attn_bwd_dq_kernel<KEPT, HP, NPAN, W, G>
                    : a.drop.thresh ? attn_bwd_dq_kernel<MADE, HP, NPAN, W, G>
                                    : attn_bwd_dq_kernel<NODROP, HP, NPAN, W, G>;
        return attn_go(kern, seq, W * 32, nbh, W * HP * G * 64, attn_lds<HP, NPAN, W, G>(true, false), a, st);
    }
};
struct attn_dkv_launch {
    template <int HP, int NPAN, int W, int G> static int go(int seq, int nbh, const AttnArgs& a, hipStream_t st) {
        auto kern = a.keep ? attn_bwd_dkv_kernel<KEPT, HP, NPAN, W, G>
                    : a.drop.thresh ? attn_bwd_dkv_kernel<MADE, HP, NPAN, W, G>
                                    : attn_bwd_dkv_kernel<NODROP, HP, NPAN, W, G>;
        // 128-wide heads: a block per half
        return attn_go(kern, seq, W * 32, nbh * NPAN, W * HP * G * 64, attn_lds<HP, NPAN, W, G>(true, true), a, st);
    }
};
// Both backward kernels go in one launch where their grids together are at most a round and a quarter of the blocks that the chip holds,
// under a causal mask two and a quarter, for its short blocks fill in behind the long ones; 128-wide heads, which make scores twice, a
// round and a round and three quarters.  Else one after the other.  Each alone is bound by its longest walk while at most half of the
// chip has work; together they take the longer of the two instead of the sum, and a launch less.  What it costs is delta a second time,
// by every dK / dV block for the queries it will meet, and registers: beyond these lines both weigh more than what overlaps.
// A round is what waves and LDS let in: eight waves a CU; one block of four where two rings fill more than half of LDS (64-wide heads,
// two waves in two groups).  Heads stay on their XCD, so uneven ones leave empty blocks in the grid, which go to no other XCD: they count
// (three heads are on three XCDs, 96 CUs).  Rounds: one after the other / together, us (heads, keys; D: with dropout).  The bits are the same.
//   padding   64-wide 2x4   1.1: 41.9 / 36.0 (7, 1114 D)   1.25: 38.2 / 34.3 (5, 1268 D)   1.4: 34.2 / 42.9 (1, 1377)   2: 44.8 / 57.1 (2, 1997)
//             2x2   1.25: 21.4 / 18.5 (16, 640)   1.7: 41.3 / 51.3 (5, 1682)      4x2   1.6: 56.2 / 63.9 (12, 1549)
//             4x1   1.1: 69.0 / 63.4 (19, 1499)   1.7: 53.2 / 50.8 (46, 1116)     pairs 2x2   1.1: 31.6 / 26.5 (2, 1066)   1.3: 39.7 / 46.8 (3, 1323)
//   no mask   64-wide 4x1   1.1: 65.2 / 56.8 (25, 1070)   1.5: 115.0 / 114.7 (24, 1934)   pairs 2x1   1.1: 25.3 / 22.1 (46, 366)
//   causal    64-wide 2x4   1.9: 41.4 / 37.3 (3, 1938)    4x1   1.9: 88.0 / 77.0 (28, 1897)    4x2   1.6: 54.1 / 42.3 (16, 1575)
//             2x2   2: 30.8 / 27.0 (16, 987)   2.4: 32.6 / 33.2 (9, 1153)   3: 39.9 / 47.3 (10, 1500)
//             pairs 2x2   2.25: 35.1 / 33.1 (12, 1112)   2x1   2.1: 90.6 / 78.8 (17, 1402 D)   2.3: 42.5 / 43.8 (34, 919)
//   128-wide  4x1   no mask 0.9: 88.0 / 90.0 (14, 1182)   1.1: 88.3 / 106.4 (20, 1055)   padding 0.9: 43.9 / 37.6 (37, 420 D)
//             4x1   causal 1.6: 58.7 / 58.8 (54, 628)   2.2: 85.6 / 90.0 (51, 874)
//             4x2   padding 1: 158 / 122 (2, 1973 D)   causal 1.7: 48.1 / 43.4 (27, 629)
static constexpr int kOwnDeltaSeq = 2048;    // longest sequence whose deltas a block keeps in LDS
struct attn_bwd_launch {
    template <int HP, int NPAN, int W, int G> static int go(int seq, int nbh, const AttnArgs& a, hipStream_t st) {
        constexpr size_t dq_lds = attn_lds<HP, NPAN, W, G>(true, false), dkv_lds = attn_lds<HP, NPAN, W, G>(true, true);
        constexpr size_t own_at = dkv_lds > dq_lds ? dkv_lds : dq_lds;
        constexpr int waves = W * HP * G;
        constexpr unsigned round = waves == 4 && own_at > 80 * 1024 ? 256 : 256 * 8 / waves;
        const unsigned dkv = attn_grid(seq, W * 32, nbh * NPAN), dq = attn_grid(seq, W * 32, nbh);
        const unsigned quarters = NPAN == 2 ? (a.mask == BB_MASK_CAUSAL ? 7 : 4) : (a.mask == BB_MASK_CAUSAL ? 9 : 5);
        const bool room = dkv + dq <= round / 4 * quarters;
        if (seq > kOwnDeltaSeq || !room) {
            // the dQ kernel first: it also leaves delta = rowsum(dO o O) of its queries for the dK / dV kernel
            const int rc = attn_dq_launch::go<HP, NPAN, W, G>(seq, nbh, a, st);
            return rc ? rc : attn_dkv_launch::go<HP, NPAN, W, G>(seq, nbh, a, st);
        }
        const size_t lds = own_at + (size_t)HP * ((seq + 63) / 64 * 64) * sizeof(float);
        auto kern = a.keep ? attn_bwd_kernel<KEPT, HP, NPAN, W, G>
                    : a.drop.thresh ? attn_bwd_kernel<MADE, HP, NPAN, W, G>
                                    : attn_bwd_kernel<NODROP, HP, NPAN, W, G>;
        BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, lds));
        bb_launch(kern, dim3(dkv + dq), dim3(W * HP * G * 64), lds, st, a, (int)dkv, (int)own_at);
        BB_LAUNCH_CHECK();
        return BB_OK;
    }
};
// The shape of a block (waves W of 32 rows x groups G), by the number of blocks of 128 rows and the length of the walk.  Device time in us:
//                                         forward, W x G                        backward
//   blocks, heads                  4x1   4x2   2x4   2x2   2x1           4x1   4x2   2x4   2x2   2x1
//    24  1 x 2,   1500 causal     25.7  22.3  14.9  17.4  25.6          46.9  39.2  30.1  33.0  48.1
//    32  2 x 4,    512 causal     11.3  10.6   7.7   8.2  10.8          19.5  18.3  14.6  14.7  18.1
//   128  2 x 8,   1024 causal     18.8  16.9  11.5  12.8  18.7          33.9  29.4  27.8  25.7  34.3
//   128  4 x 16,   200 causal      7.3   7.2   6.3   6.2   6.6          12.9  13.2  16.8  14.2  12.1
//   150  2 x 25,   300 padding     8.0   8.2  11.0   7.7   8.0          16.6  22.7  24.0  18.2  15.5
//   192  1 x 12,  2043 padding    29.2  25.2  31.3  23.3  36.0          67.5  63.2  78.5  87.3   110
//   240  3 x 10,  1000 causal     19.0  17.0  16.2  13.7  19.2          36.8  40.5  42.2  40.9  38.3
//   256  4 x 16,   512 causal     11.8  11.1  12.7   9.1  11.4          23.1  28.3  34.1  30.7  23.7
//   320  2 x 20,  1024 causal     19.7  18.3  22.1  14.9  19.7          49.2  45.3  58.2  55.6  49.2
//   352  1 x 22,  2000 causal     34.0  29.8  34.8  25.1  34.8          84.5  70.5  85.6  91.9  86.1
//   384  8 x 12,   512 causal     12.6  13.0  18.8  13.9  12.8          32.7  42.7  51.7  46.8  33.7
//   384  4 x 12,  1024 padding    22.5  23.4  31.3  26.5  23.2          61.5  76.3  80.0  82.7  60.6
//   400  1 x 25,  2048 causal     57.4  55.3  65.5  49.5  73.9           118   104   129   148   121      (dropout)
//   512  8 x 16,   512 causal     13.3  13.6  24.0  15.3  13.6          34.1  47.8  68.6  61.4  37.6
//    96  6 x 8,    175, no mask    6.6                     6.2          11.0                    10.4
//   128  2 x 8,   1024, no mask   18.5                    18.6          33.4                    34.2
// Few blocks want their walks shared by groups, and small blocks, which also even out long and short walks under a causal mask; the
// backward, whose waves look ahead by themselves, only where the walk is long, and it loses the launch that both passes share.  Of
// 65 to 128 blocks (backward, share of the time of two waves in four groups that do not look ahead, by 4x1, 2x2, 2x4): causal, 224 to 447
// keys 0.84 0.83 0.93, with dropout kept 0.73 0.63 0.69, 640 to 899 1.03 0.82 0.82 and 0.86 0.63 0.62, 1200 to 1535 1.21 0.94 0.92 and 0.94 0.69
// 0.62, 1800 to 2048 1.31 0.93 0.84; padding, 224 to 447 0.81 0.82 0.91, 640 to 899 1.00 0.95 0.96 and with dropout 0.79 0.77 0.75, 1200 to 1535 1.07
// 1.01 0.95, dropout made again 1.10 1.04 0.92, 1800 to 2048 1.38 1.03 0.95.
// Heads of 128 find room for two groups: 4 heads, 1024 causal with dropout (32) 41.6 118.9 / 33.9 86.4.  Pairs of heads have twice the
// waves: two a head in two groups (a walk of both heads by two waves in four groups / this: 1 x 4 pairs, 500 causal 9.6 16.4 / 8.3 15.3,
// 2 x 4, 300, padding, dropout 9.6 20.7 / 7.8 17.0; four waves in two groups / four a head: 4 x 8, 512 causal 10.6 24.8 / 9.2 22.4); else
// two a head, blocks as small as those of four waves of one head, for one block of eight waves a CU stands still at every barrier (four
// a head / two, forward and backward with kept decisions: 8 x 8 pairs, 128, dropout 8.9 11.2 / 6.6 9.6; 4 x 8, 1020, dropout 41.4 73.1 / 40.5 72.0,
// causal 40.7 73.4 / 29.4 57.1; decisions made again, 7 x 7, 1633 226 559 / 182 455, causal 130 322 / 89 226, padding 163 389 / 127 336, without
// dropout 81 213 / 74 197).
// Attention without a mask keeps the one walk.  Groups add the same terms in another order: as near the exact sums as before, but
// not the same last bits, and the stage that ends the reference's script (no mask; a LayerNorm whose rows are summed up, which
// cancels to 1e-4 of its terms) passes gradients on in which such bits show as 3 to 5 %.
template <typename L, int HP, int NPAN> static int attn_shape(int seq, int nbh, const AttnArgs& a, hipStream_t st) {
    const int64_t blocks = (int64_t)nbh * ((seq + 127) / 128);
    const bool masked = a.mask != BB_MASK_NONE;
    if constexpr (HP == 2) {
        if (masked && blocks <= 128 && seq >= 160) return L::template go<HP, NPAN, 2, 2>(seq, nbh, a, st);
        return L::template go<HP, NPAN, 2, 1>(seq, nbh, a, st);
    } else if constexpr (NPAN == 2) {
        if (masked && blocks <= 256 && seq >= 448) return L::template go<HP, NPAN, 4, 2>(seq, nbh, a, st);
    } else if constexpr (std::is_same_v<L, attn_fwd_launch>) {
        if (masked && seq >= 160) {
            if (blocks <= 128) return L::template go<HP, NPAN, 2, 4>(seq, nbh, a, st);
            if (blocks <= 256 || (blocks <= 400 && seq >= 1024 && a.mask == BB_MASK_CAUSAL)) return L::template go<HP, NPAN, 2, 2>(seq, nbh, a, st);
        }
        if (blocks <= 128 && seq <= 320) return L::template go<HP, NPAN, 2, 1>(seq, nbh, a, st);
    } else {
        if (masked && seq >= 1536 && blocks > 128 && blocks <= 400) return L::template go<HP, NPAN, 4, 2>(seq, nbh, a, st);
        if (masked && blocks > 64 && blocks <= 128) {
            if (seq >= (a.drop.thresh ? 640 : 1200)) return L::template go<HP, NPAN, 2, 4>(seq, nbh, a, st);
            if (seq >= (a.mask == BB_MASK_CAUSAL ? 224 : 448)) return L::template go<HP, NPAN, 2, 2>(seq, nbh, a, st);
        }
        if (masked && seq >= 320 && blocks <= 64) return L::template go<HP, NPAN, 2, 4>(seq, nbh, a, st);
        if (blocks <= 128 && seq <= 320) return L::template go<HP, NPAN, 2, 1>(seq, nbh, a, st);
    }
    if constexpr (HP == 1) return L::template go<HP, NPAN, 4, 1>(seq, nbh, a, st);
}
template <typename L> static int attn_launch(int head_dim, int seq, int batch, int heads, const AttnArgs& a, hipStream_t st) {
    if (head_dim == 128) return attn_shape<L, 1, 2>(seq, batch * heads, a, st);
    if (head_dim == 64) return attn_shape<L, 1, 1>(seq, batch * heads, a, st);
    return attn_shape<L, 2, 1>(seq, batch * (heads / 2), a, st);    // pairs of heads
}

static int attention_fwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q,
                                const void* k, const void* v, int64_t ld_qkv, void* out, int64_t ld_out, float* lse,
                                const int32_t* key_len, float dropout_p, uint32_t dropout_k0, uint32_t dropout_k1,
                         uint32_t* keep, void* stream) {
    int rc = check_attn("bb_attention_fwd", dtype, mask, batch, heads, seq, head_dim, ld_qkv, ld_out, key_len);
    if (rc) return rc;
    if (batch == 0 || seq == 0) return BB_OK;
    BB_REQUIRE(q && k && v && out && lse, "bb_attention_fwd: null pointer");
    BB_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "bb_attention_fwd: dropout_p must be in [0, 1)");
    BB_REQUIRE((uintptr_t)keep % 128 == 0, "bb_attention_fwd: keep must be aligned to 128 bytes");
    AttnArgs a = {};
    a.drop = bb_drop_key(dropout_p, dropout_k0, dropout_k1, (uint64_t)batch * heads * (uint64_t)seq * (uint64_t)seq);
    a.keep = a.drop.thresh ? (uint32_t*)keep : nullptr;
    a.q = (const bf16*)q; a.k = (const bf16*)k; a.v = (const bf16*)v;
    a.out = (bf16*)out; a.lse = lse; a.key_len = key_len;
    a.ld_qkv = ld_qkv; a.ld_o = ld_out;
    a.batch = batch; a.heads = heads; a.seq = seq; a.mask = mask;
    a.scale = 1.0f / sqrtf((float)head_dim);
    a.scale_log2 = a.scale * 1.4426950408889634f;
    return attn_launch<attn_fwd_launch>(head_dim, seq, batch, heads, a, (hipStream_t)stream);
}

static int attention_bwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q,
                                const void* k, const void* v, int64_t ld_qkv, const void* out, const void* d_out,
                                int64_t ld_out, const float* lse, float* delta, void* dq, void* dk, void* dv,
                                int64_t ld_dqkv, const int32_t* key_len, float dropout_p, uint32_t dropout_k0,
                                uint32_t dropout_k1, const uint32_t* keep, void* stream) {
    int rc = check_attn("bb_attention_bwd", dtype, mask, batch, heads, seq, head_dim, ld_qkv, ld_out, key_len);
    if (rc) return rc;
    if (batch == 0 || seq == 0) return BB_OK;
    BB_REQUIRE(q && k && v && out && d_out && lse && delta && dq && dk && dv, "bb_attention_bwd: null pointer");
    BB_REQUIRE(ld_dqkv % 4 == 0 && ld_dqkv >= heads * head_dim, "bb_attention_bwd: bad gradient leading dimension");
    BB_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "bb_attention_bwd: dropout_p must be in [0, 1)");
    BB_REQUIRE((uintptr_t)keep % 128 == 0, "bb_attention_bwd: keep must be aligned to 128 bytes");
    AttnArgs a = {};
    a.drop = bb_drop_key(dropout_p, dropout_k0, dropout_k1, (uint64_t)batch * heads * (uint64_t)seq * (uint64_t)seq);
    a.keep = a.drop.thresh ? (uint32_t*)keep : nullptr;
    a.q = (const bf16*)q; a.k = (const bf16*)k; a.v = (const bf16*)v;
    a.o = (const bf16*)out; a.d_o = (const bf16*)d_out;
    a.dq = (bf16*)dq; a.dk = (bf16*)dk; a.dv = (bf16*)dv;
    a.lse = (float*)lse; a.delta = delta; a.key_len = key_len;
    a.ld_qkv = ld_qkv; a.ld_o = ld_out; a.ld_dqkv = ld_dqkv;
    a.batch = batch; a.heads = heads; a.seq = seq; a.mask = mask;
    a.scale = 1.0f / sqrtf((float)head_dim);
    a.scale_log2 = a.scale * 1.4426950408889634f;
    return attn_launch<attn_bwd_launch>(head_dim, seq, batch, heads, a, (hipStream_t)stream);
}

extern "C" int64_t bb_attention_keep_words(int batch, int heads, int seq) { return (int64_t)batch * heads * keep_blocks(seq) * 32; }
extern "C" int bb_attention_fwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k, const void* v,
                                int64_t ld_qkv, void* out, int64_t ld_out, float* lse, const int32_t* key_len, float dropout_p,
                                uint32_t dropout_k0, uint32_t dropout_k1, void* stream) {
    return attention_fwd(dtype, mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, out, ld_out, lse, key_len, dropout_p, dropout_k0,
                         dropout_k1, nullptr, stream);
}
extern "C" int bb_attention_fwd_keep(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k,
                                     const void* v, int64_t ld_qkv, void* out, int64_t ld_out, float* lse, const int32_t* key_len,
                                     float dropout_p, uint32_t dropout_k0, uint32_t dropout_k1, uint32_t* keep, void* stream) {
    return attention_fwd(dtype, mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, out, ld_out, lse, key_len, dropout_p, dropout_k0,
                         dropout_k1, keep, stream);
}
extern "C" int bb_attention_bwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k, const void* v,
                                int64_t ld_qkv, const void* out, const void* d_out, int64_t ld_out, const float* lse, float* delta,
                                void* dq, void* dk, void* dv, int64_t ld_dqkv, const int32_t* key_len, float dropout_p,
                                uint32_t dropout_k0, uint32_t dropout_k1, void* stream) {
    return attention_bwd(dtype, mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, out, d_out, ld_out, lse, delta, dq, dk, dv, ld_dqkv,
                         key_len, dropout_p, dropout_k0, dropout_k1, nullptr, stream);
}
extern "C" int bb_attention_bwd_keep(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k,
                                     const void* v, int64_t ld_qkv, const void* out, const void* d_out, int64_t ld_out, const float* lse,
                                     float* delta, void* dq, void* dk, void* dv, int64_t ld_dqkv, const int32_t* key_len, float dropout_p,
                                     uint32_t dropout_k0, uint32_t dropout_k1, const uint32_t* keep, void* stream) {
    return attention_bwd(dtype, mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, out, d_out, ld_out, lse, delta, dq, dk, dv, ld_dqkv,
                         key_len, dropout_p, dropout_k0, dropout_k1, keep, stream);
}
