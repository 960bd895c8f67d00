// Staging of an int8 convolution's input: NCHW (int8, or fp32 quantized on the way) -> [n][hs][ws][cp] int8 with halo.
#pragma once
#include "tsx_common.hpp"

namespace tsx {

struct StageGeom {
    int n, c, h, w;        // source NCHW
    int hs, ws, cp;        // staged extent
    int pad_top, pad_left;
    int pad_value;         // int8 halo value
};

// Whether stage_planes takes the layer (a channel plane of at least four elements).
bool stage_planes_takes(const StageGeom &g);
// scales == nullptr: src is int8 and copied; otherwise fp32, quantized as cpu::Quantize does at the element's index.
int stage_planes(const StageGeom &g, const void *src, const float *scales, int n_scales, int64_t group_len, int64_t bulk8, int8_t *xs,
                 hipStream_t stream);

}  // namespace tsx
