// Internal interface of the fp32 convolution kernel of large layers (conv2d_f32_window.hip), used by gemm_f32.hip.
#pragma once
#include "tsx_common.hpp"

namespace tsx {

// One layer's geometry and operands; a matrix product [cout][c] x [c][wo] is the 1x1 layer n = ho = h = 1.
struct ConvF32Layer {
    int n, c, h, w, cout, kh, kw, pad_top, pad_left, stride_h, stride_w, dil_h, dil_w, ho, wo;
    const float *x_dev, *w_dev;
};

// The tile (and patch form) the kernel would take for the layer, -1 where it cannot, and the cycles expected of the busiest
// CU (0: the tile is forced); its extents; the launch.
int conv_f32_window_tile(const ConvF32Layer &l, double *cycles = nullptr);
void conv_f32_window_tile_size(int tile, int *rows, int *positions);
int conv_f32_window(const ConvF32Layer &l, int tile, const float *bias, int act, float slope, float padding_value, float *out,
                    hipStream_t stream);

}  // namespace tsx
