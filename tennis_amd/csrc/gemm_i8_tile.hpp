// int8 GEMM on tiles of 128 x 128, 128 x 256 or 256 x 256 outputs (gemm_i8_tile.hip).
#pragma once
#include "igemm_i8.hpp"

namespace tsx {

struct GemmTileParams : EpiParams {
    const int8_t *xs;    // activations [m][pitch] at any alignment, at least 16 bytes; cp: the columns rounded up to 64
    const int8_t *wp;    // weights as tsx_gemm_i8_pack_weights lays them out
    int m, cout, coutp, cp, cblocks, pitch;
    int row_tiles, col_tiles, tiles_per_xcd;   // set by the launch
};

// The tile this kernel should take the problem on, or 0: another kernel.  1: 128 x 128, 2: 128 x 256, 3: 256 x 256.
// unpadded: rows of another length or alignment than the other kernels read.
int gemm_i8_tile_choose(int m, int n, int k, bool int8_out, bool unpadded);
// The epilogue must hold no residual, no staged output and not the exact Mish, and its quantize groups must be rows; n and k
// below 2^23.
int gemm_i8_tile_launch(const GemmTileParams &p, int tile, hipStream_t stream);

#ifdef __HIPCC__
// ---- activation rows read where they are
// The kernels read K in pieces of 16 bytes and steps of 64.  Rows of another length need no padded copy: what a piece holds
// behind its row's end -- the next row's first bytes -- meets weights that are zero.  Only a piece that would end behind the
// whole matrix (the last row's last ones) is read earlier, so that it ends with the matrix, and shifted into place.
// Loads at any alignment cost the vector memory path an extra line now and then; the copy cost a launch and a memory round
// trip, 3.5 us of the 13 .. 17 us of 197 rows, K = 1500.
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));

__device__ __forceinline__ v4i load_piece(const int8_t *at) { return *reinterpret_cast<const v4i_any *>(at); }

// bytes s .. 15 of a piece to its front (s > 15: all of it lies behind the matrix, any value does)
__device__ __forceinline__ v4i shift_piece(v4i v, int s) {
    if (s & 8) v = v4i{v[2], v[3], 0, 0};
    if (s & 4) v = v4i{v[1], v[2], v[3], 0};
    const unsigned b = unsigned(s) & 3u;
    return v4i{int(__builtin_amdgcn_alignbyte(unsigned(v[1]), unsigned(v[0]), b)), int(__builtin_amdgcn_alignbyte(unsigned(v[2]), unsigned(v[1]), b)),
               int(__builtin_amdgcn_alignbyte(unsigned(v[3]), unsigned(v[2]), b)), int(__builtin_amdgcn_alignbyte(0u, unsigned(v[3]), b))};
}

// emit() of a GEMM's element: the quantize group is the row, as long as the reference's float arithmetic does not round the
// group length (emit divides 64 bits by 64 bits for each element: 300 x 3000, K = 3000, 17.2 us with fp32 and 22 with int8
// output)
__device__ __forceinline__ void emit_row(const EpiParams &p, int cout, int acc, int row, int64_t idx, float dq, float bias, float row_scale) {
    if (p.out_acc) p.out_acc[idx] = acc;
    if (!p.out_f32 && !p.out_i8) return;
    const float v = epi_value<true>(p, acc, idx, dq, bias, row_scale);
    if (p.out_f32) p.out_f32[idx] = v;
    if (p.out_i8) {
        const float s = p.n_qscales == 1 ? p.q_scales[0] : p.q_scales[p.q_group_len == cout ? row : idx / p.q_group_len];
        p.out_i8[idx] = int8_t(quantize_value(__fmul_rn(v, s), p.n_qscales == 1 && idx < p.q_bulk8));
    }
}
#endif

}  // namespace tsx
