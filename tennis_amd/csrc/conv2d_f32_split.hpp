// Internal interface of the fp32 convolution on the bf16 matrix cores (conv2d_f32_split.hip), used by gemm_f32.hip.
#pragma once
#include "gemm_f32.hpp"

namespace tsx {

struct ConvF32Split {
    int tile;                 // -1: no tile suits the layer
    size_t workspace_bytes;
    double us;                // expected; 0: the tile is forced
    int slices;               // of the input channels, each a workgroup's of its own
};
ConvF32Split conv_f32_split_choose(const ConvF32Layer &l, size_t workspace_bytes);      // the fastest that fits
void conv_f32_split_tile_size(int tile, int *rows, int *positions, int *patch);      // patch: cells it is built for
int conv_f32_split(const ConvF32Layer &l, const ConvF32Split &choice, const float *bias, int act, float slope, float padding_value, float *out,
                   void *workspace, hipStream_t stream);

}  // namespace tsx
