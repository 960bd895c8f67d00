#include "conv2d_i8_pt_kernel.hpp"

namespace tsx {
template <>
int pt_launch_layer<2, 9, 1, 4>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<2, 9, 1, 4, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<2, 9, 1, 4, false>(p, grid, lds_bytes, stream);
}
template <>
int pt_launch_layer<2, 9, 2, 4>(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    return p.act == TSX_ACT_MISH ? pt_launch_kernel<2, 9, 2, 4, true>(p, grid, lds_bytes, stream) : pt_launch_kernel<2, 9, 2, 4, false>(p, grid, lds_bytes, stream);
}
}  // namespace tsx
