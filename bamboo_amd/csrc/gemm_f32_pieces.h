// fp32 products on bf16 matrix instructions (gemm_f32_pieces.hip): which problems take them, on which tiles.
#pragma once
#include "gemm_kernels.h"

enum PiecesTile { P_NONE = 0, P128x128, P128x64 };
PiecesTile pick_pieces(const bb_gemm_desc* descs, int count);   // several: weight gradients that share a launch, on 128x128 tiles
int launch_pieces(GemmArgs& g, int layout, PiecesTile tile, hipStream_t st);
int launch_pieces_grouped(GroupedArgs& G, hipStream_t st);
