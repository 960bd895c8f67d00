// The int8 convolution of 1x1 layers as streams of pixels (conv2d_i8_px.hip).
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

// Whether the kernel serves the layer (WsPlan::px); whether it also writes the epilogue and reaches the tensors of a call;
// launch.  g holds the extents of the buffer that is read; the weights are packed as for the layer's other kernels.
void px_plan(const WsGeom &g, WsPlan *pl);
bool px_joins(const WsGeom &g);      // whether a residual may join
bool px_takes(const WsGeom &g, const WsPlan &pl, const EpiParams &ep);
int px_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream);

}  // namespace tsx
