#include "conv2d_i8_pt_kernel.hpp"

namespace tsx {
template <>
int pt_launch_layer<1, 9, 1, 5>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<1, 9, 1, 5, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<1, 9, 1, 5, false>(p, grid, lds_bytes, stream);
}
template <>
int pt_launch_layer<1, 9, 2, 5>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<1, 9, 2, 5, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<1, 9, 2, 5, false>(p, grid, lds_bytes, stream);
}
template <>
int pt_launch_layer<1, 6, 1, 3>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<1, 6, 1, 3, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<1, 6, 1, 3, false>(p, grid, lds_bytes, stream);
}
template <>
int pt_launch_layer<1, 6, 2, 3>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<1, 6, 2, 3, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<1, 6, 2, 3, false>(p, grid, lds_bytes, stream);
}
}  // namespace tsx
