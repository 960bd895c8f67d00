// int8 GEMM on tiles of 128 x 128, 128 x 256 or 256 x 256 outputs (gemm_i8_tile.hip).
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

struct GemmTileParams : EpiParams {
    const int8_t *xs;    // activations [m][cp], 16-byte aligned, cp a multiple of 64 with zeros behind k
    const int8_t *wp;    // weights as tsx_gemm_i8_pack_weights lays them out
    int m, cout, coutp, cp, cblocks;
    int row_tiles, col_tiles, tiles_per_xcd;   // set by the launch
};

// The tile this kernel should take the problem on, or 0: another kernel.  1: 128 x 128, 2: 128 x 256, 3: 256 x 256.
int gemm_i8_tile_choose(int m, int n, int k, bool int8_out);
// The epilogue must hold no residual, no staged output and not the exact Mish, and its quantize groups must be rows; n and k
// below 2^23.
int gemm_i8_tile_launch(const GemmTileParams &p, int tile, hipStream_t stream);

}  // namespace tsx
