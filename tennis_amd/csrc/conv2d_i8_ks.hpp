// The int8 convolution with K split over a workgroup's wavefronts (conv2d_i8_ks.hip).
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

// Chooses a tile for the layer (WsPlan::ks, 0: another kernel); reads weights packed as ws_pack_weights packs them and
// writes every epilogue.
void ks_plan(const WsGeom &g, WsPlan *pl);
int ks_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream);

}  // namespace tsx
