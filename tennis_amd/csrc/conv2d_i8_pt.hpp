// The int8 convolution of layers of several taps on few channels as streams of small tiles (conv2d_i8_pt.hip).
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

// Whether the kernel serves the layer, and its tile (WsPlan::pt); whether it also writes the epilogue and reaches the tensors of a
// call; launch.  g holds the extents of the buffer that is read; the weights are packed as for the layer's other kernels.
void pt_plan(const WsGeom &g, WsPlan *pl);
bool pt_takes(const WsGeom &g, const WsPlan &pl, const EpiParams &ep);
int pt_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream);

}  // namespace tsx
