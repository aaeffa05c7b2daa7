// fp32 products on bf16 matrix instructions (gemm_f32_pieces.hip): which problems take them, on which tiles.
#pragma once
#include "gemm_kernels.h"

// Longer fp32 contractions: problems with fewer than two 64x64 tiles per CU and at least 16 k-tiles take 64x32 tiles whose contraction two groups of
// two waves share: twice the tiles to deal to the CUs, each wave's chain of matrix instructions as long as before.  NT and NN
// only: the weight gradients (TN) of a layer share a grouped launch.
inline bool pick_f32_split(int M, int N, int K, int64_t batches, int layout) {
    return layout != BB_TN && (int64_t)((M + 63) / 64) * ((N + 63) / 64) * batches < 2 * 256 && K >= 512;
}

enum PiecesTile { P_NONE = 0, P128x128, P128x64 };
PiecesTile pick_pieces(const bb_gemm_desc* descs, int count);   // several: weight gradients that share a launch, on 128x128 tiles
int launch_pieces(GemmArgs& g, int layout, PiecesTile tile, hipStream_t st);
int launch_pieces_grouped(GroupedArgs& G, hipStream_t st);
