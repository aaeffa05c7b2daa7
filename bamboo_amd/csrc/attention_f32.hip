// Masked softmax-attention for gfx950, fp32, heads of 32, 64 or 128 columns, with the probabilities kept: one kernel for the
// forward pass, two for the backward pass.
//
// Stands in for MultiHeadedAttention.attention of the reference (DeepSpeedExamples/pipeline_parallelism/transformer.py:117-127)
// and its autograd backward, in the precision and with the kept probabilities of the batched products and row kernels
// (gemm_f32.h, softmax_{fwd,bwd}_kernel) that run every other shape.  Those against this, us, forward / backward: 4 x 12 heads
// of 64, 512 positions, causal 71 / 121 -> 33 / 56, unmasked 72 / 121 -> 44 / 77 (a large product's rate would be 24 / 49);
// 4 heads of 64 and 64 positions 17 / 33 -> 6.5 / 11, with dropout 29 / 54 -> 7 / 13.  The error of the gradients against 64 bits
// at 512 positions went from 4.4e-7 to 2.5e-7 (shorter chains), below 128 positions it is what it was.
//
// What bounds it: fp32 matrix instructions (64 cycles each) on large batches, the chain of launches on small ones.  So nothing is
// made twice -- the backward pass reads the kept probabilities instead of making them again, a fifth of whose cost at 64 columns
// would be two more products -- and key tiles that the mask rules out are neither multiplied nor read.  A block owns 32 queries
// and keeps their scores in LDS, so the softmax and its derivative see whole rows without a pass over memory of their own.
// Operands go from memory straight into registers: a fragment of 8 KB lasts 2048 matrix cycles, the loads need no staging.
#include "common.h"

struct AttnF32Args {
    const float* q; const float* k; const float* v;   // head 0 of batch 0; row stride ld_qkv
    const float* d_o;                                 // backward: gradient of the context, row stride ld_o
    float* out;                                       // forward: context, row stride ld_o
    float* prob;                                      // [batch, heads, seq, seq], in front of dropout
    float* d_score;                                   // backward scratch, as prob: gradient of the scaled scores
    float* dq; float* dk; float* dv;                  // row stride ld_dqkv
    const int32_t* key_len;
    int64_t ld_qkv, ld_o, ld_dqkv;
    int batch, heads, seq, mask;
    float scale;                                      // 1 / sqrt(d)
    DropKey drop;                                     // dropout on the probabilities (thresh 0: none)
};
template <> struct BbDropAt<AttnF32Args> { static constexpr int32_t value = offsetof(AttnF32Args, drop); };
template <> struct BbPointersAt<AttnF32Args> : BbPointerRun<11> {};   // q .. key_len
static_assert(offsetof(AttnF32Args, ld_qkv) == 11 * sizeof(void*), "BbPointersAt<AttnF32Args>");

constexpr int kMaxLd = 1 << 19;   // floats: kMaxSeq rows of fewer are less than 2^31 bytes
constexpr int kWaves = 8;
constexpr int kMaxSeq = 1024;   // 32 rows of scores: 132 of a CU's 160 KB of LDS
// floats per row of the score strip: four past a multiple of 32, so that eight neighbouring rows start on different banks
__host__ __device__ constexpr int strip_ld(int seq) { return (seq + 31) / 32 * 32 + 4; }
static size_t strip_bytes(int seq) {
    const size_t s = (size_t)32 * strip_ld(seq) * sizeof(float), parts = kWaves * 32 * 32 * sizeof(float);
    return s > parts ? s : parts;
}

// block -> (rank, batch * head): whole (batch, head) pairs to an XCD (their K and V stay in its L2), rank 0 first
struct F32BlockMap { int rank, bh; };
__device__ __forceinline__ F32BlockMap f32_map_block(int nbh) {
    const int per_xcd = (nbh + 7) >> 3, xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    return {j / per_xcd, (j % per_xcd) * 8 + xcd};
}
// keys that query q of sample b may see; 0: none, and then every score is the mask's -1e9 and all keys get the same share
__device__ __forceinline__ int f32_limit(const AttnF32Args& a, int len, int q) {
    if (a.mask == BB_MASK_CAUSAL) return min(a.seq, q + 1);
    return len;
}
// 32-wide key tiles that a block of queries from q0 on has to look at
__device__ __forceinline__ int f32_key_tiles(const AttnF32Args& a, int len, int q0) {
    int end = a.mask == BB_MASK_CAUSAL ? q0 + 32 : len;
    if (end <= 0) end = a.seq;
    return (min(end, a.seq) + 31) / 32;
}
// A wave adds its products over keys or queries up in chains of 32 where there are at most 128 of them, of 128 beyond (a chain's
// end costs a sixteenth of 32's matrix time); as a mask of the count of 32-wide pieces.
__device__ __forceinline__ int f32_chain(int seq) { return seq <= 128 ? 0 : 3; }
__device__ __forceinline__ int f32_sample_len(const AttnF32Args& a, int b) {
    return a.mask == BB_MASK_KEY_PADDING ? max(0, min(a.seq, a.key_len[b])) : a.seq;
}
// Rows of a matrix, read through a buffer descriptor: a lane's offset in a vector register, the row in a scalar one, so that a
// load costs the matrix cores no vector instruction, and what lies past the last row reads as zero.  No load stands behind a
// branch: at a merge the compiler would wait for all that are in flight.  The kernels count on the zeros (a ragged sequence is read
// up to 31 rows past its end), and with that on the range check of a raw buffer taking the scalar offset in, also where that
// alone lies beyond the end.  So it does on gfx950: of a range of 1000 bytes inside a larger allocation, all 3509 words past it read
// as zero, 3392 of them under a scalar offset beyond it (step 100 bytes, up to 6300).
struct Rows {
    __amdgpu_buffer_rsrc_t desc;
    unsigned ld;   // bytes
    __device__ __forceinline__ Rows(const float* base, int rows, int64_t row_stride, int cols)
        : desc(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, ((unsigned)(rows - 1) * (unsigned)row_stride + cols) * 4, 0x00020000)), ld((unsigned)row_stride * 4) {}
    __device__ __forceinline__ float load1(unsigned lane, unsigned row) const {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(desc, lane, row * ld, 0));
    }
    __device__ __forceinline__ f32x4 load4(unsigned lane, unsigned row) const {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(desc, lane, row * ld, 0));
    }
};
// keep-and-scale factor of probability idx; 32-bit arithmetic where the indices fit it
__device__ __forceinline__ float f32_keep(const DropKey& d, uint64_t idx) {
    const uint32_t x = d.small ? bb_dropout_pair_bits32(d.k0, d.k1, (uint32_t)idx >> 1) : bb_dropout_pair_bits(d.k0, d.k1, idx >> 1);
    return (idx & 1 ? x >> 16 : x & 0xffffu) >= d.thresh ? d.scale : 0.f;
}
// four neighbours from an even idx on: two hashes
__device__ __forceinline__ void f32_drop4(const DropKey& d, uint64_t idx, f32x4& v) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const uint32_t x = d.small ? bb_dropout_pair_bits32(d.k0, d.k1, ((uint32_t)idx >> 1) + e) : bb_dropout_pair_bits(d.k0, d.k1, (idx >> 1) + e);
        v[2 * e] *= bb_keep_even(x, d.thresh) ? d.scale : 0.f;
        v[2 * e + 1] *= bb_keep_odd(x, d.thresh) ? d.scale : 0.f;
    }
}

// Forward: scores = Q K^T / sqrt(d), P = softmax(scores) -> prob, context = dropout(P) V.
// BWD: dP = dropout'(dO V^T), dS = P (dP - rowsum(dP P)) -> d_score, dQ = dS K / sqrt(d).
// A product of rows into the strip (eight waves take key tiles in turn; a tile's contraction in slices of 32, whose sums are
// added in order), a pass over the strip's rows (sixteen lanes a row, the row in registers), the strip times the keys' rows (waves take 32-wide
// column tiles and share the keys; the shares are added in order).  An operand
// register is loaded again as soon as its product is issued: what is in flight is a whole tile, in one set of registers.
template <int D, bool BWD>
__global__ __launch_bounds__(kWaves * 64, D == 128 ? 2 : 4) void attn_f32_rows_kernel(const AttnF32Args a) {
    constexpr int NC = D / 8, DT = D / 32, SHARES = kWaves / DT;
    extern __shared__ __attribute__((aligned(16))) float strip[];
    __shared__ float stat[kWaves][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, half = lane >> 5;
    const F32BlockMap bm = f32_map_block(a.batch * a.heads);
    if (bm.bh >= a.batch * a.heads) return;
    const int qb = (a.seq + 31) / 32 - 1 - bm.rank;   // the late query blocks, which see most keys, first
    const int b = bm.bh / a.heads, head = bm.bh % a.heads, q0 = qb * 32;
    const int64_t row0 = (int64_t)b * a.seq;
    const int len = f32_sample_len(a, b), tiles = f32_key_tiles(a, len, q0), ld = strip_ld(a.seq);
    const float* rows_q = (BWD ? a.d_o + row0 * a.ld_o : a.q + row0 * a.ld_qkv) + head * D;
    const float* rows_k = (BWD ? a.v : a.k) + row0 * a.ld_qkv + head * D;
    const int64_t ld_q = BWD ? a.ld_o : a.ld_qkv;
    const int my_q = min(q0 + col, a.seq - 1);
    const uint64_t row_of_prob = (uint64_t)bm.bh * a.seq;

    // ---- scores of a tile, transposed: lane = query, registers = keys.  Contraction in pairs (8 c + i, 8 c + 4 + i).
    {
        f32x4 x[NC], y[NC];
        const Rows keys(rows_k, a.seq, a.ld_qkv, D), queries(rows_q, a.seq, ld_q, D);
        const unsigned at_key = col * keys.ld + 16 * half, at_query = col * queries.ld + 16 * half;
        const auto fetch = [&](int t, int u) {
#pragma unroll
            for (int c = 4 * u; c < 4 * u + 4; ++c) x[c] = keys.load4(at_key + 32 * c, t * 32);
            __builtin_amdgcn_sched_barrier(0);   // issued here, not in a burst in front of the next tile
        };
        if (wave < tiles) {
#pragma unroll
            for (int c = 0; c < NC; ++c) y[c] = queries.load4(at_query + 32 * c, q0);
#pragma unroll
            for (int u = 0; u < DT; ++u) fetch(wave, u);
        }
        float mx = -INFINITY;
        const int limit = f32_limit(a, len, my_q);
        for (int t = wave; t < tiles; t += kWaves) {
            const int key0 = t * 32 + 4 * half;
            f32x16 s;
            const int next = min(t + kWaves, tiles - 1);
#pragma unroll
            for (int u = 0; u < DT; ++u) {
                f32x16 part;
#pragma unroll
                for (int r = 0; r < 16; ++r) part[r] = 0.f;
#pragma unroll
                for (int c = 4 * u; c < 4 * u + 4; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i) part = __builtin_amdgcn_mfma_f32_32x32x2f32(x[c][i], y[c][i], part, 0, 0, 0);
                fetch(next, u);
                if (u == 0) s = part;
                else {
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] += part[r];
                }
            }
            if constexpr (!BWD) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] *= a.scale;
                if (t * 32 + 32 > (a.mask == BB_MASK_CAUSAL ? q0 + 1 : len)) {   // some query may not see some key
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = key0 + 8 * (r >> 2) + (r & 3);
                        s[r] = key >= a.seq ? -INFINITY : key < limit ? s[r] : -1e9f;
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
            }
            float* o = strip + col * ld + key0;
#pragma unroll
            for (int g = 0; g < 4; ++g) *(f32x4*)(o + 8 * g) = f32x4{s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
        }
        if constexpr (!BWD) {
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            if (half == 0) stat[wave][col] = mx;
        }
    }
    __syncthreads();

    // ---- rows: sixteen lanes each, 16 bytes a lane and step, the row in registers.  Forward, the strip keeps exp(score - max),
    // dropped out: the context is divided by the row's sum at its end.
    {
        const int row = wave * 4 + (lane >> 4), q = q0 + row, sub = (lane & 15) * 4, end = tiles * 32;
        const uint64_t base = (row_of_prob + min(q, a.seq - 1)) * a.seq;
        float* s = strip + row * ld + sub;
        constexpr int STEPS = kMaxSeq / 64;
        f32x4 v[STEPS];
        const auto drop = [&](f32x4& x, int i) {
            if (a.drop.thresh) f32_drop4(a.drop, base + i * 64 + sub, x);
        };
        float sum = 0.f, inv;
        if constexpr (!BWD) {
            float mx = stat[0][row];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, stat[w][row]);
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (i * 64 < end && i * 64 + sub < end) {
                    v[i] = *(const f32x4*)(s + i * 64);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] = expf(v[i][e] - mx);
                    sum += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
                    f32x4 kept = v[i];
                    drop(kept, i);
                    *(f32x4*)(s + i * 64) = kept;
                }
        } else {
            // what lies past the sequence has no probability
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (i * 64 < end) {
                    v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (i * 64 + sub < a.seq) v[i] = *(const f32x4*)(a.prob + base + i * 64 + sub);
                }
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (i * 64 < end && i * 64 + sub < end) {
                    f32x4 dp = *(const f32x4*)(s + i * 64);
                    if (a.drop.thresh) {
                        drop(dp, i);
                        *(f32x4*)(s + i * 64) = dp;
                    }
                    sum += (v[i][0] * dp[0] + v[i][1] * dp[1]) + (v[i][2] * dp[2] + v[i][3] * dp[3]);
                }
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
        if constexpr (!BWD) {
            inv = 1.0f / sum;
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (i * 64 < end && i * 64 + sub < min(end, a.seq) && q < a.seq)
                    *(f32x4*)(a.prob + base + i * 64 + sub) = f32x4{v[i][0] * inv, v[i][1] * inv, v[i][2] * inv, v[i][3] * inv};
            if (q < a.seq)
                for (int k = end + sub; k < a.seq; k += 64) *(f32x4*)(a.prob + base + k) = f32x4{0.f, 0.f, 0.f, 0.f};
            __syncthreads();
            if ((lane & 15) == 0) stat[0][row] = inv;
        } else {
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (i * 64 < end && i * 64 + sub < end) {
                    f32x4 ds = *(const f32x4*)(s + i * 64);
#pragma unroll
                    for (int e = 0; e < 4; ++e) ds[e] = v[i][e] * (ds[e] - sum);
                    *(f32x4*)(s + i * 64) = ds;
                    if (i * 64 + sub < a.seq && q < a.seq) *(f32x4*)(a.d_score + base + i * 64 + sub) = ds;
                }
        }
    }
    __syncthreads();

    // ---- strip x rows of the keys: lane = column, registers = queries
    const int dt = wave % DT, share = wave / DT;
    const Rows w((BWD ? a.k : a.v) + row0 * a.ld_qkv + head * D + dt * 32, a.seq, a.ld_qkv, 32);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (share < tiles) {
        float x[16];
        const unsigned at = col * 4 + 4 * half * w.ld;
        const auto fetch_rows = [&](int t, int c) {   // rows 8 c + 4 half + {0..3} of the tile
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * c + i] = w.load1(at, t * 32 + 8 * c + i);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int c = 0; c < 4; ++c) fetch_rows(share, c);
        f32x16 part;
        int n = 0;
        const int chain = f32_chain(a.seq);
        for (int t = share; t < tiles; t += SHARES) {
            if ((n++ & chain) == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[r] = n == 1 ? 0.f : acc[r] + part[r];
                    part[r] = 0.f;
                }
            }
            const float* p = strip + col * ld + t * 32 + 4 * half;
            f32x4 s[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) s[c] = *(const f32x4*)(p + 8 * c);
            const int next = min(t + SHARES, tiles - 1);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma unroll
                for (int i = 0; i < 4; ++i) part = __builtin_amdgcn_mfma_f32_32x32x2f32(s[c][i], x[4 * c + i], part, 0, 0, 0);
                fetch_rows(next, c);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += part[r];
    }
    // the shares meet in LDS; each wave finishes its part of the registers
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) strip[(share * DT + dt) * 1024 + r * 64 + lane] = acc[r];
    __syncthreads();
    float* o = (BWD ? a.dq + row0 * a.ld_dqkv : a.out + row0 * a.ld_o) + head * D + dt * 32 + col;
    const int64_t ld_out = BWD ? a.ld_dqkv : a.ld_o;
    constexpr int NR = 16 / SHARES;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int r = share * NR + j, row = 8 * (r >> 2) + 4 * half + (r & 3);
        float v = strip[dt * 1024 + r * 64 + lane];
#pragma unroll
        for (int p = 1; p < SHARES; ++p) v += strip[(p * DT + dt) * 1024 + r * 64 + lane];
        if (q0 + row < a.seq) o[(int64_t)(q0 + row) * ld_out] = v * (BWD ? a.scale : stat[0][row]);
    }
}

// dV = dropout(P)^T dO and dK = dS^T Q / sqrt(d): a block owns 32 keys of a head, a wave one 32-wide column tile of one of the two
// and, where that leaves waves, a share of the queries (every SHARES-th 32 of them; the shares are added in
// order).  Queries in front of a causal block's keys and padded keys contribute nothing.
template <int D>
__global__ __launch_bounds__(kWaves * 64, 4) void attn_f32_keys_kernel(const AttnF32Args a) {
    constexpr int DT = D / 32, SHARES = kWaves / (2 * DT), NQ = 16;   // pairs of queries a step
    __shared__ float parts[kWaves][16 * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, half = lane >> 5;
    const bool is_dk = wave & 1;
    const int dt = (wave >> 1) % DT, share = (wave >> 1) / DT;
    const F32BlockMap bm = f32_map_block(a.batch * a.heads);
    if (bm.bh >= a.batch * a.heads) return;
    const int b = bm.bh / a.heads, head = bm.bh % a.heads, key0 = bm.rank * 32;   // early keys, which most queries see, first
    const int64_t row0 = (int64_t)b * a.seq;
    const int len = f32_sample_len(a, b);
    const int first = a.mask == BB_MASK_CAUSAL ? key0 : 0;
    const int steps = a.mask == BB_MASK_KEY_PADDING && len > 0 && key0 >= len ? 0 : (a.seq - first + 2 * NQ - 1) / (2 * NQ);
    const uint64_t base = (uint64_t)bm.bh * a.seq * a.seq;
    const int key = min(key0 + col, a.seq - 1);
    const Rows xs((is_dk ? a.d_score : a.prob) + base, a.seq, a.seq, a.seq);
    const Rows ys((is_dk ? a.q + row0 * a.ld_qkv : a.d_o + row0 * a.ld_o) + head * D + dt * 32, a.seq, is_dk ? a.ld_qkv : a.ld_o, 32);
    const unsigned x_off = half * xs.ld + key * 4, y_off = half * ys.ld + col * 4;
    const bool drop = !is_dk && a.drop.thresh != 0;

    f32x16 acc, part;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = part[r] = 0.f;
    float x[NQ], y[NQ];
    const auto fetch = [&](int i, int j) {
        const int q = first + i * 2 * NQ + 2 * j;
        x[j] = xs.load1(x_off, q);
        y[j] = ys.load1(y_off, q);
        __builtin_amdgcn_sched_barrier(0);   // issued here, not in a burst in front of the next step
    };
    if (share < steps) {
#pragma unroll
        for (int j = 0; j < NQ; ++j) fetch(share, j);
        int n = 0;
        const int chain = f32_chain(a.seq);
        for (int i = share; i < steps; i += SHARES) {
            if ((n++ & chain) == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[r] += part[r];
                    part[r] = 0.f;
                }
            }
            const int next = min(i + SHARES, steps - 1), q0 = first + i * 2 * NQ;
            if (drop) {
#pragma unroll
                for (int j = 0; j < NQ; ++j) x[j] *= f32_keep(a.drop, base + (uint64_t)(q0 + 2 * j + half) * a.seq + key);
            }
#pragma unroll
            for (int j = 0; j < NQ; ++j) {
                part = __builtin_amdgcn_mfma_f32_32x32x2f32(x[j], y[j], part, 0, 0, 0);
                fetch(next, j);
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += part[r];
    }
    // the shares meet in LDS; each wave finishes its part of the registers
    float* o = (is_dk ? a.dk : a.dv) + row0 * a.ld_dqkv + head * D + dt * 32 + col;
    const float f = is_dk ? a.scale : 1.0f;
    constexpr int NR = 16 / SHARES;
    if constexpr (SHARES > 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) parts[wave][r * 64 + lane] = acc[r];
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int r = share * NR + j, k = key0 + 8 * (r >> 2) + 4 * half + (r & 3);
        float v = acc[j];
        if constexpr (SHARES > 1) {
            const int w = wave % (2 * DT);
            v = parts[w][r * 64 + lane];
#pragma unroll
            for (int p = 1; p < SHARES; ++p) v += parts[w + p * 2 * DT][r * 64 + lane];
        }
        if (k < a.seq) o[(int64_t)k * a.ld_dqkv] = v * f;
    }
}

// =========================================================================================
// host entry points
// =========================================================================================
// Where the batched products are the better ones still, they stay: 128-wide heads of more than 256 positions in so few blocks
// that each CU has at most one and two thirds have none -- its eight waves then work through more columns than the products'
// smaller tiles do (us, products / this, forward + backward: 1 head of 512 68 / 77, 4 heads 76 / 77, 12 heads 162 / 95 causal;
// 1 head of 256 56 / 50).  Longer sequences: their strip finds no room.
extern "C" int bb_attention_probs_supported(int dtype, int batch, int heads, int seq, int head_dim) {
    if (dtype != BB_F32 || batch <= 0 || heads <= 0 || seq <= 0 || seq % 4 != 0 || seq > kMaxSeq) return 0;
    if (head_dim != 32 && head_dim != 64 && head_dim != 128) return 0;
    if (3 * (int64_t)heads * head_dim >= kMaxLd) return 0;
    return head_dim != 128 || seq <= 256 || (int64_t)batch * heads * ((seq + 31) / 32) >= 96;
}

static int check_probs(const char* name, int dtype, int mask, int batch, int heads, int seq, int head_dim, int64_t ld_qkv,
                       int64_t ld_o, const int32_t* key_len, float dropout_p) {
    BB_REQUIRE(dtype == BB_F32 && heads > 0 && (head_dim == 32 || head_dim == 64 || head_dim == 128) && seq > 0 && seq % 4 == 0 && seq <= kMaxSeq,
               "%s: fp32, heads of 32, 64 or 128 columns, a sequence length that is a multiple of 4 and at most %d (got dtype %d, %d "
               "heads of %d, %d positions)", name, kMaxSeq, dtype, heads, head_dim, seq);
    BB_REQUIRE(mask >= BB_MASK_NONE && mask <= BB_MASK_KEY_PADDING, "%s: bad mask %d", name, mask);
    BB_REQUIRE(mask != BB_MASK_KEY_PADDING || key_len, "%s: key_padding mask needs key_len", name);
    BB_REQUIRE(batch >= 0, "%s: bad shape", name);
    BB_REQUIRE(ld_qkv < kMaxLd && ld_o < kMaxLd, "%s: leading dimension too large", name);
    BB_REQUIRE(ld_qkv % 4 == 0 && ld_o % 4 == 0 && ld_qkv >= (int64_t)heads * head_dim && ld_o >= (int64_t)heads * head_dim, "%s: bad leading dimension", name);
    BB_REQUIRE(((int64_t)batch * heads + 8) * ((seq + 31) / 32) < (1ll << 31), "%s: batch * heads * seq exceeds the grid limit", name);
    BB_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "%s: dropout_p must be in [0, 1)", name);
    return BB_OK;
}
static unsigned probs_grid(int seq, int nbh) { return (unsigned)(8 * ((nbh + 7) / 8) * ((seq + 31) / 32)); }
static AttnF32Args probs_args(int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k, const void* v,
                              int64_t ld_qkv, void* prob, const int32_t* key_len, float p, uint32_t k0, uint32_t k1) {
    AttnF32Args a = {};
    a.drop = bb_drop_key(p, k0, k1, (uint64_t)batch * heads * (uint64_t)seq * (uint64_t)seq);
    a.q = (const float*)q; a.k = (const float*)k; a.v = (const float*)v;
    a.prob = (float*)prob;
    a.key_len = key_len;
    a.ld_qkv = ld_qkv;
    a.batch = batch; a.heads = heads; a.seq = seq; a.mask = mask;
    a.scale = (float)(1.0 / sqrt((double)head_dim));
    return a;
}
template <int D, bool BWD> static int launch_rows(const AttnF32Args& a, hipStream_t st) {
    const size_t lds = strip_bytes(a.seq);
    auto kern = attn_f32_rows_kernel<D, BWD>;
    BB_HIP_CHECK(bb_allow_dynamic_lds((const void*)kern, lds));
    bb_launch(kern, dim3(probs_grid(a.seq, a.batch * a.heads)), dim3(kWaves * 64), lds, st, a);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
template <int D> static int launch_keys(const AttnF32Args& a, hipStream_t st) {
    bb_launch((attn_f32_keys_kernel<D>), dim3(probs_grid(a.seq, a.batch * a.heads)), dim3(kWaves * 64), 0, st, a);
    BB_LAUNCH_CHECK();
    return BB_OK;
}
static bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }

extern "C" int bb_attention_probs_fwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k,
                                      const void* v, int64_t ld_qkv, void* out, int64_t ld_out, void* prob, const int32_t* key_len,
                                      float dropout_p, uint32_t dropout_k0, uint32_t dropout_k1, void* stream) {
    int rc = check_probs("bb_attention_probs_fwd", dtype, mask, batch, heads, seq, head_dim, ld_qkv, ld_out, key_len, dropout_p);
    if (rc) return rc;
    if (batch == 0) return BB_OK;
    BB_REQUIRE(q && k && v && out && prob, "bb_attention_probs_fwd: null pointer");
    BB_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(prob), "bb_attention_probs_fwd: operands must be 16-byte aligned");
    AttnF32Args a = probs_args(mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, prob, key_len, dropout_p, dropout_k0, dropout_k1);
    a.out = (float*)out;
    a.ld_o = ld_out;
    hipStream_t st = (hipStream_t)stream;
    return head_dim == 32 ? launch_rows<32, false>(a, st) : head_dim == 64 ? launch_rows<64, false>(a, st) : launch_rows<128, false>(a, st);
}

extern "C" int bb_attention_probs_bwd(int dtype, int mask, int batch, int heads, int seq, int head_dim, const void* q, const void* k,
                                      const void* v, int64_t ld_qkv, const void* d_out, int64_t ld_out, const void* prob, void* d_score,
                                      void* dq, void* dk, void* dv, int64_t ld_dqkv, const int32_t* key_len, float dropout_p,
                                      uint32_t dropout_k0, uint32_t dropout_k1, void* stream) {
    int rc = check_probs("bb_attention_probs_bwd", dtype, mask, batch, heads, seq, head_dim, ld_qkv, ld_out, key_len, dropout_p);
    if (rc) return rc;
    if (batch == 0) return BB_OK;
    BB_REQUIRE(q && k && v && d_out && prob && d_score && dq && dk && dv, "bb_attention_probs_bwd: null pointer");
    BB_REQUIRE(ld_dqkv >= (int64_t)heads * head_dim, "bb_attention_probs_bwd: bad gradient leading dimension");
    BB_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(d_out) && aligned16(prob) && aligned16(d_score),
               "bb_attention_probs_bwd: operands must be 16-byte aligned");
    AttnF32Args a = probs_args(mask, batch, heads, seq, head_dim, q, k, v, ld_qkv, (void*)prob, key_len, dropout_p, dropout_k0, dropout_k1);
    a.d_o = (const float*)d_out;
    a.ld_o = ld_out;
    a.d_score = (float*)d_score;
    a.dq = (float*)dq; a.dk = (float*)dk; a.dv = (float*)dv;
    a.ld_dqkv = ld_dqkv;
    hipStream_t st = (hipStream_t)stream;
    rc = head_dim == 32 ? launch_rows<32, true>(a, st) : head_dim == 64 ? launch_rows<64, true>(a, st) : launch_rows<128, true>(a, st);
    if (rc) return rc;
    return head_dim == 32 ? launch_keys<32>(a, st) : head_dim == 64 ? launch_keys<64>(a, st) : launch_keys<128>(a, st);
}
