// Sums of partial rows that the blocks of an earlier launch left behind (the gain and shift gradients of LayerNorms), in a fixed
// order whichever kernel adds them up: one of their own, or the weight gradients' launch with a few blocks more in front.
#pragma once

#include "common.h"

constexpr int RED_WAVES = 16;

// Sum of partial rows p = first, first + step, ... in that order, eight loads in flight at a time.
__device__ __forceinline__ float sum_partials(const float* __restrict__ src, int first, int step, int nparts, int64_t stride) {
    float s = 0.f;
    int p = first;
    for (; p + 7 * step < nparts; p += 8 * step) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = src[(int64_t)(p + j * step) * stride];
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[j];
    }
    if (p < nparts) {   // the last few go out together as well
        float v[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) v[j] = p + j * step < nparts ? src[(int64_t)(p + j * step) * stride] : 0.f;
#pragma unroll
        for (int j = 0; j < 7; ++j) s += v[j];
    }
    return s;
}

// out0[i] / out1[i] += sum over p < nparts of partial[p][0 / 1][i], i < n
constexpr int PARTIAL_SUMS_MAX = BB_PARTIAL_SUMS_MAX;
struct PartialSums {
    const float* partial[PARTIAL_SUMS_MAX];
    float* out0[PARTIAL_SUMS_MAX];
    float* out1[PARTIAL_SUMS_MAX];
    int nparts[PARTIAL_SUMS_MAX], n[PARTIAL_SUMS_MAX], first_block[PARTIAL_SUMS_MAX + 1];
    int count;
    int blocks;   // a multiple of 8, so that the blocks behind them keep their XCDs
};
template <> struct BbPointersAt<PartialSums> : BbPointerRun<3 * PARTIAL_SUMS_MAX> {};   // partial, out0, out1
static_assert(offsetof(PartialSums, nparts) == 3 * PARTIAL_SUMS_MAX * sizeof(void*), "BbPointersAt<PartialSums>");

// One block owns 64 columns of one of the two outputs.  Sixteen interleaved shares of the partial rows (p = w, w+16, ...) are summed
// by its WAVES waves, 16 / WAVES each, and the sixteen results combined in order: no bit depends on WAVES.  red: [RED_WAVES][64].
template <int WAVES> __device__ __forceinline__ void partial_sums_block(const PartialSums& a, int b, float* red) {
    if (b >= a.first_block[a.count]) return;
    int r = 0;
    while (r + 1 < a.count && b >= a.first_block[r + 1]) ++r;
    b -= a.first_block[r];
    const int n = a.n[r], nb = (n + 63) / 64, which = b >= nb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = (b - which * nb) * 64 + lane;
    const float* src = a.partial[r] + (int64_t)which * n + i;
    for (int w = wave; w < RED_WAVES; w += WAVES) red[w * 64 + lane] = i < n ? sum_partials(src, w, RED_WAVES, a.nparts[r], (int64_t)2 * n) : 0.f;
    __syncthreads();
    if (wave == 0 && i < n) {
        float s = red[lane];
#pragma unroll
        for (int w = 1; w < RED_WAVES; ++w) s += red[w * 64 + lane];
        float* out = which ? a.out1[r] : a.out0[r];
        out[i] += s;
    }
}

// checked (elementwise.hip)
int bb_partial_sums_args(const char* who, const bb_partial_sums* sums, int count, PartialSums& a);
// whether no two of them add into the same memory: the blocks of a launch add without atomics
bool bb_partial_sums_apart(const bb_partial_sums* sums, int count);
