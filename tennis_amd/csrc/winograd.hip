// Winograd F(6x6, 3x3) and F(2x2, 3x3) fp32 convolution, restating
// Conv2dWinogradAlgorithm<float>::winograd_f63 / winograd_f23
// (src/kernels/cpu/winograd_algorithm.cpp:504-947 / :57-459) with the padding rule of
// KernelCommonFunc::in_out_pad_and_fix_size (src/kernels/common/function.cpp:14-78).
// F(6,3) is described below; F(2,3) is its twin with 4x4 patches (stride 2), 16 frequencies and
// transforms made of sums and differences only.
//
//   U = G g G^T      kernel transform, once per weight tensor
//   V = B^T d B      input transform of every 8x8 patch (stride 6)
//   M_f = U_f V_f    64 independent GEMMs (Cout x Cin x tiles)
//   Y = A^T M A      output transform, cut to the true output size       -> out NCHW
//
// F(6,3) in fp32 amplifies single roundings to ~1e-5 of an O(1) output, the same size as the
// parity tolerance, so this path reproduces the reference's arithmetic exactly instead of merely
// approximating it:
//   * every transform uses the reference's factoring AND its fused multiply-adds: the reference
//     is built with gcc -O3 -mfma, whose default contraction fuses a*b+c patterns (in
//     a*c1 - b*c2 it fuses the first product and rounds the second); those FMAs are written
//     out explicitly here and the file is compiled with -ffp-contract=off;
//   * the GEMMs accumulate like the reference's pack8/kernel_8x8 micro-kernel
//     (src/kernels/cpu/math_cpu.cpp:386-700): one k-ascending FMA chain per output, and for
//     columns beyond an image's last full block of 8 four interleaved chains combined as
//     (s0+s1), (s2+s3), 0+s01, +s23.  v_mfma_f32_32x32x2_f32 IS such a chain: every output is
//     fma(a1, b1, fma(a0, b0, c)) with one rounding per step and denormals kept (compared with
//     fmaf on the host, bit for bit, over normal, widely scaled and denormal operands), so the
//     matrix cores give the reference's bits as long as a step carries k and k + 1 in order.
//
// Layouts.  A "column" is one tile of one image.  The columns an image computes as plain chains (its
// first tiles/8*8) come first, image after image, padded to whole fragments of 32; then the rest
// ("tail" columns), padded likewise.  U and V are stored as MFMA operands: [frequency][fragment of 32
// rows or columns][group t of 8 channels][lane][4], lane l's element j being channel 8t + 2j + l/32 of row or
// column l%32 -- one contiguous KiB per four MFMA steps, loaded straight into registers (no LDS: with 64 cycles
// per MFMA the operands of a 32 x 64 tile need a quarter of the CU's load path).  M is [frequency][cout][columns].
// Channels beyond Cin are -0 in U and +0 in V: their product -0 leaves every accumulator as it is, signed zeros
// included.
#include "tsx_common.hpp"

#include <algorithm>

namespace tsx {
namespace {

// U and V are float arrays to the caller: 16- and 8-byte accesses at any float's address (the instructions are the same)
typedef float v2f __attribute__((ext_vector_type(2), aligned(4)));
typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------- transforms (explicit FMAs)

__device__ __forceinline__ void bt_row(const float *i0, float *o) {
    // winograd_algorithm.cpp:640-663 (first pass over the rows of the patch)
    o[0] = fmaf(i0[4] - i0[2], 5.25f, i0[0] - i0[6]);
    o[7] = fmaf(i0[3] - i0[5], 5.25f, i0[7] - i0[1]);
    const float tmp12_a = fmaf(-i0[4], 4.25f, i0[2] + i0[6]);
    const float tmp12_b = fmaf(-i0[3], 4.25f, i0[1] + i0[5]);
    o[1] = tmp12_a + tmp12_b;
    o[2] = tmp12_a - tmp12_b;
    const float tmp34_a = fmaf(-i0[4], 1.25f, fmaf(i0[2], 0.25f, i0[6]));
    const float tmp34_b = fmaf(i0[5], 2.f, fmaf(i0[1], 0.5f, -(i0[3] * 2.5f)));
    o[3] = tmp34_a + tmp34_b;
    o[4] = tmp34_a - tmp34_b;
    const float tmp56_a = fmaf(fmaf(-i0[4], 1.25f, i0[2]), 4.f, i0[6]);
    const float tmp56_b = fmaf(i0[5], 0.5f, fmaf(i0[1], 2.f, -(i0[3] * 2.5f)));
    o[5] = tmp56_a + tmp56_b;
    o[6] = tmp56_a - tmp56_b;
}

__device__ __forceinline__ void bt_col(const float *d, float *o) {
    // winograd_algorithm.cpp:668-692 (second pass; tmp12_b's operand order differs from the first)
    o[0] = fmaf(d[4] - d[2], 5.25f, d[0] - d[6]);
    o[7] = fmaf(d[3] - d[5], 5.25f, d[7] - d[1]);
    const float tmp12_a = fmaf(-d[4], 4.25f, d[2] + d[6]);
    const float tmp12_b = fmaf(-d[3], 4.25f, d[1]) + d[5];
    o[1] = tmp12_a + tmp12_b;
    o[2] = tmp12_a - tmp12_b;
    const float tmp34_a = fmaf(-d[4], 1.25f, fmaf(d[2], 0.25f, d[6]));
    const float tmp34_b = fmaf(d[5], 2.f, fmaf(d[1], 0.5f, -(d[3] * 2.5f)));
    o[3] = tmp34_a + tmp34_b;
    o[4] = tmp34_a - tmp34_b;
    const float tmp56_a = fmaf(fmaf(-d[4], 1.25f, d[2]), 4.f, d[6]);
    const float tmp56_b = fmaf(d[5], 0.5f, fmaf(d[1], 2.f, -(d[3] * 2.5f)));
    o[5] = tmp56_a + tmp56_b;
    o[6] = tmp56_a - tmp56_b;
}

__device__ __forceinline__ void at_pass(const float *t, float *o) {
    // winograd_algorithm.cpp:775-795 / :808-830; every multiplier is a power of two, so fused
    // and unfused forms round identically -- only the left-to-right order of the sums matters.
    const float re0 = t[1] + t[2];
    const float re1 = t[1] - t[2];
    const float re2 = t[3] + t[4];
    const float re3 = t[3] - t[4];
    const float re4 = t[5] + t[6];
    const float re5 = t[5] - t[6];
    o[0] = t[0] + re0 + re2 + re4 * 32.f;
    o[1] = re1 + re3 + re3 + re5 * 16.f;
    o[2] = re0 + re2 * 4 + re4 * 8.f;
    o[3] = re1 + re3 * 8 + re5 * 4.f;
    o[4] = re0 + re2 * 16 + re4 + re4;
    o[5] = re1 + re3 * 32 + re5 + t[7];
}


struct WinoGeom {
    int n, c, h, w, cout, ho, wo, pad_top, pad_left, th, tw, tiles;
    float padding_value;
    int rfrags, kgroups;       // 32-row fragments of U, groups of 8 channels
    int n8, mfrags, nfrags;    // chain columns per image, their fragments, all fragments
    int cols;                  // 32 * nfrags: the row pitch of M
};

// The image and tile of a column; false for the columns that pad a fragment.
__device__ __forceinline__ bool column_tile(const WinoGeom &g, int col, int &img, int &tile) {
    const bool tail = col >= g.mfrags * 32;
    const int c = tail ? col - g.mfrags * 32 : col, per = tail ? g.tiles - g.n8 : g.n8;
    img = per > 0 ? c / per : 0;
    tile = c - img * per + (tail ? g.n8 : 0);
    return per > 0 && img < g.n;
}

// Element (channel, row or column) -> float index inside one frequency of U or V
__device__ __forceinline__ int64_t operand_index(int frag, int kgroups, int t, int lane, int j) {
    return ((int64_t(frag) * kgroups + t) * 64 + lane) * 4 + j;
}

// U = G g G^T, one thread per (cout, cin) of the padded operand (TILE 6: winograd_algorithm.cpp:504-566, TILE 2:
// :57-105, before their pack8_A).
template <int TILE>
__global__ __launch_bounds__(256) void wino_kernel_transform_kernel(const float *__restrict__ w, int cout, int cin, int rfrags,
                                                                   int kgroups, float *__restrict__ u) {
    constexpr int P = TILE + 2;
    const int64_t per_f = int64_t(rfrags) * kgroups * 256;
    const int64_t id = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= per_f) return;
    const int j = int(id % 4), lane = int(id / 4 % 64), t = int(id / 256 % kgroups), rf = int(id / 256 / kgroups);
    const int co = rf * 32 + lane % 32, ci = 8 * t + 2 * j + lane / 32;
    if (co >= cout || ci >= cin) {
        for (int f = 0; f < P * P; ++f) u[f * per_f + id] = -0.f;
        return;
    }
    const float G6[8][3] = {{1.0f, 0.0f, 0.0f},
                            {-2.f / 9, -2.f / 9, -2.f / 9},
                            {-2.f / 9, 2.f / 9, -2.f / 9},
                            {1.f / 90, 1.f / 45, 2.f / 45},
                            {1.f / 90, -1.f / 45, 2.f / 45},
                            {1.f / 45, 1.f / 90, 1.f / 180},
                            {1.f / 45, -1.f / 90, 1.f / 180},
                            {0.0f, 0.0f, 1.0f}};
    const float G2[4][3] = {{1.f, 0.f, 0.f}, {0.5f, 0.5f, 0.5f}, {0.5f, -0.5f, 0.5f}, {0.f, 0.f, 1.f}};
    float g[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) g[i] = w[(int64_t(co) * cin + ci) * 9 + i];
    float tmp[3][P];
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const float *G = TILE == 6 ? G6[i] : G2[i % 4];
            tmp[r][i] = fmaf(g[r * 3 + 2], G[2], fmaf(g[r * 3 + 0], G[0], g[r * 3 + 1] * G[1]));
        }
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const float *G = TILE == 6 ? G6[i] : G2[i % 4];
            u[(i * P + q) * per_f + id] = fmaf(tmp[2][q], G[2], fmaf(tmp[0][q], G[0], tmp[1][q] * G[1]));
        }
}

// V of F(6,3).  One workgroup = the 32 columns of a fragment x four channels of one parity of a channel group (a
// lane then owns whole 16-byte operand elements); thread (i, column) transforms row i of the column's four patches,
// the rows cross to columns through LDS, and it transforms column i and stores its eight frequencies.  One thread
// per patch, as before, is under one wavefront per SIMD on 8 images of 28x28x256 and waits for its 64 loads alone:
// 9.2 us there.
constexpr int WT_CH = 4;      // channels per workgroup

__global__ __launch_bounds__(256) void wino_input_transform_kernel(const float *__restrict__ x, WinoGeom g, float *__restrict__ v) {
    __shared__ float rows[WT_CH][8][8][32];
    const int i = threadIdx.x / 32, lc = threadIdx.x % 32;
    const int frag = blockIdx.x, t = blockIdx.y / 2, hf = blockIdx.y % 2;
    int img, tile;
    const bool valid = column_tile(g, frag * 32 + lc, img, tile);
    if (!valid) img = tile = 0;                              // a padding column: loads tile 0, result never used
    const int ty = tile / g.tw, tx = tile - ty * g.tw;
    const int hh = ty * 6 + i - g.pad_top, w0 = tx * 6 - g.pad_left;
    const bool row_in = hh >= 0 && hh < g.h;
    const float *src = x + int64_t(img) * g.c * g.h * g.w + min(max(hh, 0), g.h - 1) * g.w;
    float d[WT_CH][8];
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        const float *plane = src + int64_t(min(8 * t + 2 * q + hf, g.c - 1)) * g.h * g.w;
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) d[q][jj] = plane[min(max(w0 + jj, 0), g.w - 1)];
    }
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        // outside the tensor: the conv padding and the bottom/right fill both use padding_value
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) d[q][jj] = (row_in && w0 + jj >= 0 && w0 + jj < g.w) ? d[q][jj] : g.padding_value;
        float o[8];
        bt_row(d[q], o);
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) rows[q][i][jj][lc] = o[jj];
    }
    __syncthreads();
    float o[WT_CH][8];
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        float col[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) col[r] = rows[q][r][i][lc];
        bt_col(col, o[q]);
        if (8 * t + 2 * q + hf >= g.c) {
#pragma unroll
            for (int r = 0; r < 8; ++r) o[q][r] = 0.f;       // channel padding
        }
    }
    const int64_t per_f = int64_t(g.nfrags) * g.kgroups * 256;
    float *dst = v + operand_index(frag, g.kgroups, t, lc + 32 * hf, 0);
#pragma unroll
    for (int r = 0; r < 8; ++r) *reinterpret_cast<v4f *>(dst + (r * 8 + i) * per_f) = v4f{o[0][r], o[1][r], o[2][r], o[3][r]};
}

// V of F(2,3): B^T d B (winograd_algorithm.cpp:181-243), row combinations (i0-i2, i1+i2, i2-i1, i1-i3) first, then the
// same combination across columns, in the reference's grouping.  Thread = one column x four channels of one parity.
__global__ __launch_bounds__(256) void wino23_input_transform_kernel(const float *__restrict__ x, WinoGeom g, float *__restrict__ v) {
    const int lc = threadIdx.x % 32, part = blockIdx.y * 8 + threadIdx.x / 32;     // part = (channel group, parity)
    const int frag = blockIdx.x, t = part / 2, hf = part % 2;
    if (t >= g.kgroups) return;
    int img, tile;
    const bool valid = column_tile(g, frag * 32 + lc, img, tile);
    if (!valid) img = tile = 0;
    const int ty = tile / g.tw, tx = tile - ty * g.tw;
    const int h0 = ty * 2 - g.pad_top, w0 = tx * 2 - g.pad_left;
    const float *src = x + int64_t(img) * g.c * g.h * g.w;
    float d[4][4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float *plane = src + int64_t(min(8 * t + 2 * q + hf, g.c - 1)) * g.h * g.w;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) d[q][i][j] = plane[min(max(h0 + i, 0), g.h - 1) * g.w + min(max(w0 + j, 0), g.w - 1)];
    }
    v4f o[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool real = 8 * t + 2 * q + hf < g.c;
        float r[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = h0 + i >= 0 && h0 + i < g.h && w0 + j >= 0 && w0 + j < g.w;
                d[q][i][j] = in ? d[q][i][j] : g.padding_value;
            }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r[0][j] = d[q][0][j] - d[q][2][j];
            r[1][j] = d[q][1][j] + d[q][2][j];
            r[2][j] = d[q][2][j] - d[q][1][j];
            r[3][j] = d[q][1][j] - d[q][3][j];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            o[k * 4 + 0][q] = real ? r[k][0] - r[k][2] : 0.f;
            o[k * 4 + 1][q] = real ? r[k][1] + r[k][2] : 0.f;
            o[k * 4 + 2][q] = real ? r[k][2] - r[k][1] : 0.f;
            o[k * 4 + 3][q] = real ? r[k][1] - r[k][3] : 0.f;
        }
    }
    const int64_t per_f = int64_t(g.nfrags) * g.kgroups * 256;
    float *dst = v + operand_index(frag, g.kgroups, t, lc + 32 * hf, 0);
#pragma unroll
    for (int f = 0; f < 16; ++f) *reinterpret_cast<v4f *>(dst + f * per_f) = o[f];
}

// M_f = U_f V_f for every frequency, in the reference's accumulation order.  A wavefront computes 32 output channels x
// FN fragments of columns; the wavefronts of a workgroup take consecutive row fragments of the same columns (their V
// loads meet in L1).  Workgroups b, b + 8, ... run on one XCD: each XCD gets whole frequencies, whose U and V then
// stay in its L2 (8 x 456 KB at 8 images of 28x28x256).  RING groups of 8 channels are in flight per wavefront.
// Bound by the fp32 MFMA and by what a CU fetches besides: 1.68 GFLOP at that shape = 11 us at 157 TFLOP/s, 128 dependent MFMAs
// per wavefront.  It takes 20 .. 21 us there with its launch, from 26 .. 28 at one wavefront per SIMD, whose addresses waited
// for its MFMAs, and with the tail's 8 real columns computed as 32 (the whole convolution 41.5 -> 36.2 us; 16 images 112x112, 64 to 64
// channels, F(6,3) 156 -> 113, F(2,3) 320 -> 220; 1 image 304x304, 16 to 32, 45 -> 27 and 72 -> 33).  Chains on the vector ALUs,
// one lane per 4 x 4 outputs, took 276 + 31 us.
constexpr int WG_RING = 4;

// A fragment of U or V (T groups) as a buffer, and a lane's operand element in it.  Base and group are scalar, the lane's offset is
// constant: an address that the vector ALUs compute per load goes to registers that MFMAs in the pipe still read, and waits for
// them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t fragment_buffer(const float *base, int64_t index, int T) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base) + index * T * 256, 0, T * 1024, 0x00020000);
}
__device__ __forceinline__ v4f fragment_element(__amdgpu_buffer_rsrc_t fragment, int lane_offset, int group_offset) {
    return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(fragment, lane_offset, group_offset, 0));
}

// The four chains of the 32 x 16 outputs in s[row half] combined, and the channels left over chained behind them.
__device__ __forceinline__ void wino_tail_store(const float *__restrict__ u, const float *__restrict__ v, float *__restrict__ m, const WinoGeom &g,
                                                int f, int rf, int cf, int lane, const v16f (&s)[2]) {
    const int T = g.kgroups, q = lane / 16, i = lane % 16, k4 = g.c / 4 * 4;
    const int m8 = g.cout / 8 * 8;
    float *dst = m + int64_t(f) * g.cout * g.cols + g.mfrags * 32 + cf * 16 + i;
    // channels k4 .. c - 1, at most three: all their operands before the first use
    float ul[3][2][4] = {}, vl[3] = {};
    if (k4 < g.c)
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        const int k = min(k4 + e, g.c - 1);
        const int64_t at = int64_t(k / 8) * 256 + 128 * (k % 2) + k % 8 / 2;
        vl[e] = v[(int64_t(f) * g.nfrags + g.mfrags + cf / 2) * T * 256 + at + 4 * (16 * (cf % 2) + i)];
#pragma unroll
        for (int r = 0; r < 8; ++r) ul[e][r / 4][r % 4] = u[(int64_t(f) * g.rfrags + rf) * T * 256 + at + 4 * (16 * (r / 4) + 4 * q + r % 4)];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = rf * 32 + 16 * h + 4 * q + r;
            const float s01 = s[h][r] + s[h][4 + r], s23 = s[h][8 + r] + s[h][12 + r];
            float acc = row < m8 ? (0.f + s01) + s23 : (s01 + s[h][8 + r]) + s[h][12 + r];
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (k4 + e < g.c) acc = fmaf(ul[e][h][r], vl[e], acc);
            if (row < g.cout) dst[int64_t(row) * g.cols] = acc;
        }
}

// The tail columns: chains over k = q, q + 4, q + 8, ... (q = 0..3) up to k4 = k/4*4, their combination, then the up to
// three channels left as a chain behind it.  v_mfma_f32_16x16x1_f32 is four blocks of 16 x 16 with one multiply-add per step
// each: block q takes chain q, and a lane then holds all four chains of its outputs (accumulator 4 q + i of lane l: chain q,
// row 4 (l / 16) + i, column l % 16).  A fragment is 32 rows x 16 columns, an image leaves at
// most 7 columns here; a wavefront takes one.  (Two beside one another, which share U's operands, leave half the wavefronts to hide
// one another's loads: 78 layers took 8 % longer so, 8 images 11x11, 465 to 21 channels, F(6,3), 24.4 us for 19.6.)
__device__ __forceinline__ void wino_gemm_tail(const float *__restrict__ u, const float *__restrict__ v, float *__restrict__ m, const WinoGeom &g,
                                               int f, int rf, int cf, int lane) {
    constexpr int RING = 4;
    const int T = g.kgroups, q = lane / 16, i = lane % 16;
    // A lane loads the operand element (four channels of one parity) of its row, of the row sixteen further (+ 64 floats) and of
    // its column: the lower half-wave those of group 2 p, the upper of group 2 p + 1.  Chain q's channels 8t + q and 8t + 4 + q
    // are floats q / 2 and q / 2 + 2 of both groups: a half-wave swap each.
    // (The group is part of the lane's offset here: loads beyond the last one are then outside of the fragment's buffer.)
    const auto ua = fragment_buffer(u, int64_t(f) * g.rfrags + rf, T);
    const auto vb = fragment_buffer(v, int64_t(f) * g.nfrags + g.mfrags + cf / 2, T);
    const int row_at = 16 * (i + 32 * (q % 2)) + 1024 * (q / 2), column_at = row_at + 256 * (cf % 2);
    v16f s[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) s[0][r] = s[1][r] = 0.f;
    const int steps = g.c / 4;                               // of four channels, one to a chain
    v4f a[RING][2], b[RING];                       // [slot][row half], [slot]
    auto load = [&](auto slot, int pair) __attribute__((always_inline)) {
        constexpr int sl = decltype(slot)::value;
        a[sl][0] = fragment_element(ua, row_at + pair * 2048, 0);
        a[sl][1] = fragment_element(ua, row_at + 256 + pair * 2048, 0);
        b[sl] = fragment_element(vb, column_at + pair * 2048, 0);
    };
    auto split = [](const v4f &e, float (&of_step)[4]) __attribute__((always_inline)) {
        const auto low = __builtin_amdgcn_permlane32_swap(__float_as_int(e[0]), __float_as_int(e[1]), false, false);
        const auto high = __builtin_amdgcn_permlane32_swap(__float_as_int(e[2]), __float_as_int(e[3]), false, false);
        of_step[0] = __int_as_float(low[0]);
        of_step[1] = __int_as_float(high[0]);
        of_step[2] = __int_as_float(low[1]);
        of_step[3] = __int_as_float(high[1]);
    };
    auto multiply = [&](auto slot, int live) __attribute__((always_inline)) {      // the first `live` steps of the pair
        constexpr int sl = decltype(slot)::value;
        float ea[2][4], eb[4];
        split(a[sl][0], ea[0]);
        split(a[sl][1], ea[1]);
        split(b[sl], eb);
        static_for<0, 4>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            if (e < live) {
#pragma unroll
                for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(ea[h][e], eb[e], s[h], 0, 0, 0);
            }
        });
    };
    static_for<0, RING - 1>([&](auto sc) {
        load(sc, decltype(sc)::value);
        __builtin_amdgcn_sched_barrier(0);
    });
    int pair = 0;
    for (; 4 * (pair + RING) <= steps; pair += RING)
        static_for<0, RING>([&](auto sc) {
            constexpr int sl = decltype(sc)::value;
            load(std::integral_constant<int, (sl + RING - 1) % RING>{}, pair + sl + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(sc, 4);
            __builtin_amdgcn_sched_barrier(0);
        });
    // what is left: pairs of groups, the last perhaps of fewer steps
    static_for<0, RING>([&](auto sc) {
        constexpr int sl = decltype(sc)::value;
        if constexpr (sl == RING - 1) load(sc, pair + sl);
        multiply(sc, steps - 4 * (pair + sl));
    });
    wino_tail_store(u, v, m, g, f, rf, cf, lane, s);
}

// TAIL: and one fragment of 16 tail columns (see wino_gemm_tail) with them, whose rows are these.
template <int FN, bool TAIL>
__device__ __forceinline__ void wino_gemm_chain(const float *__restrict__ u, const float *__restrict__ v, float *__restrict__ m, const WinoGeom &g,
                                                int f, int rf, int cf0, int tf, int lane) {
    const int T = g.kgroups, q = lane / 16;
    const auto ua = fragment_buffer(u, int64_t(f) * g.rfrags + rf, T), vt = fragment_buffer(v, int64_t(f) * g.nfrags + g.mfrags + tf / 2, T);
    const int upper = q < 2 ? 0 : -1;                        // (bits selected: a choice between elements becomes an index)
    const int at = lane * 16, at_tail = (16 * (tf % 2) + lane % 16 + 32 * (q % 2)) * 16;
    v4f a[WG_RING], b[FN][WG_RING], bt[TAIL ? WG_RING : 1];
    v16f acc[FN], s[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
        for (int n = 0; n < FN; ++n) acc[n][r] = 0.f;
        if (TAIL) s[0][r] = s[1][r] = 0.f;
    }
    const int full = g.c / 8, steps = g.c / 4;               // groups without padding; the tail's steps, two to a group
    auto load = [&](auto slot, int t) __attribute__((always_inline)) {
        constexpr int sl = decltype(slot)::value;
        const int tt = min(t, T - 1) * 1024;                 // beyond the last group: its lines again, never used
        a[sl] = fragment_element(ua, at, tt);
#pragma unroll
        for (int n = 0; n < FN; ++n) b[n][sl] = fragment_element(fragment_buffer(v, int64_t(f) * g.nfrags + min(cf0 + n, g.mfrags - 1), T), at, tt);
        if constexpr (TAIL) bt[sl] = fragment_element(vt, at_tail, tt);
    };
    auto multiply = [&](auto slot, int live) __attribute__((always_inline)) {      // live: the tail's steps of this group
        constexpr int sl = decltype(slot)::value;
        // the tail's operands before the group's MFMAs: channels 8t + 4e + q of rows 0..15 and 16..31 are quarters of the
        // operand, two swaps away
        float rows[2][2], column[2];
        if constexpr (TAIL) {
            static_for<0, 2>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                const auto w = __builtin_amdgcn_permlane32_swap(__float_as_int(a[sl][2 * e]), __float_as_int(a[sl][2 * e + 1]), false, false);
                const auto r = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
                rows[e][0] = __int_as_float(r[0]);
                rows[e][1] = __int_as_float(r[1]);
                column[e] = __int_as_float((__float_as_int(bt[sl][2 * e]) & ~upper) | (__float_as_int(bt[sl][2 * e + 1]) & upper));
            });
            __builtin_amdgcn_sched_barrier(0);
        }
        auto tail_step = [&](auto ec) __attribute__((always_inline)) {
            constexpr int e = decltype(ec)::value;
            if (TAIL && e < live)
#pragma unroll
                for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(rows[e][h], column[e], s[h], 0, 0, 0);
        };
        tail_step(std::integral_constant<int, 0>{});
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < FN; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[sl][j], b[n][sl][j], acc[n], 0, 0, 0);
        tail_step(std::integral_constant<int, 1>{});
    };
    static_for<0, WG_RING - 1>([&](auto sc) {
        load(sc, decltype(sc)::value);
        __builtin_amdgcn_sched_barrier(0);                   // in the order of the loop's: what the loop waits for is counted
    });
    int t = 0;
    for (; t + WG_RING <= full; t += WG_RING)                // (no condition in here: where paths meet the compiler waits for all of them)
        static_for<0, WG_RING>([&](auto sc) {
            constexpr int sl = decltype(sc)::value;
            load(std::integral_constant<int, (sl + WG_RING - 1) % WG_RING>{}, t + sl + WG_RING - 1);
            __builtin_amdgcn_sched_barrier(0);               // left alone the scheduler sinks the loads to where they are waited for
            multiply(sc, 2);
            __builtin_amdgcn_sched_barrier(0);
        });
    static_for<0, WG_RING>([&](auto sc) {                    // the groups left over, all but the last of four in the ring already
        constexpr int sl = decltype(sc)::value;
        if constexpr (sl == WG_RING - 1) load(sc, t + sl);
        if (t + sl < T) multiply(sc, steps - 2 * (t + sl));
    });
#pragma unroll
    for (int n = 0; n < FN; ++n) {
        if (cf0 + n >= g.mfrags) break;
        float *dst = m + (int64_t(f) * g.cout + rf * 32) * g.cols + (cf0 + n) * 32 + lane % 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 8 * (r / 4) + 4 * (lane / 32) + r % 4;
            if (rf * 32 + row < g.cout) dst[int64_t(row) * g.cols] = acc[n][r];
        }
    }
    if constexpr (TAIL) wino_tail_store(u, v, m, g, f, rf, tf, lane, s);
}

// A workgroup's wavefronts are wr row fragments x wc column blocks of FN fragments.  Items are, per XCD and counted from `first`:
// row blocks of col_items of its frequencies, one frequency after the other.  The tail's fragments of 16 go with the first column
// blocks, one each (`attached`), or follow as items of their own.
// Registers for two (FN = 4) or four wavefronts per SIMD (the compiler's own choice, 267, left one).
template <int FN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(FN == 1 ? 4 : 2))) void wino_gemm_kernel(
    const float *__restrict__ u, const float *__restrict__ v, float *__restrict__ m, WinoGeom g, int wr, int wc, int row_blocks, int col_blocks,
    int tails, int attached, int rounds, int64_t first) {
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int tail_blocks = attached ? 0 : tails, col_items = (col_blocks + wc - 1) / wc, tail_items = (tail_blocks + wc - 1) / wc;
    const int64_t item = first + (blockIdx.x >> 3), chains = int64_t(rounds) * col_items * row_blocks;
    const bool tail = item >= chains;
    const int64_t at = tail ? item - chains : item;
    const int per_f = row_blocks * (tail ? tail_items : col_items), round = int(at / per_f), rest = int(at - int64_t(round) * per_f);
    const int f = (blockIdx.x & 7) + 8 * round;              // frequencies are a multiple of 8
    const int ci = rest / row_blocks, cb = ci * wc + wave / wr, rf = (rest - ci * row_blocks) * wr + wave % wr;
    if (rf >= g.rfrags || wave >= wr * wc || cb >= (tail ? tail_blocks : col_blocks)) return;
    if (tail) {
        wino_gemm_tail(u, v, m, g, f, rf, cb, lane);
    } else if (attached && cb < tails) {
        wino_gemm_chain<FN, true>(u, v, m, g, f, rf, cb * FN, cb, lane);
    } else {
        wino_gemm_chain<FN, false>(u, v, m, g, f, rf, cb * FN, 0, lane);
    }
}

// Y = A^T M A of F(6,3), cut to the true output, then the optional add_bias / activation that follow the convolution in
// the graph.  Workgroup = 32 columns x WT_CH output channels, thread (i, column): row i of M's 8x8 first, the 8x6
// intermediate crosses through LDS, then column i (i < 6).
// MISH: whether the activation may be Mish (see apply_act_basic for why that is a compile-time matter here)
template <bool MISH>
__global__ __launch_bounds__(256) void wino_output_transform_kernel(const float *__restrict__ mm, WinoGeom g,
                                                                   const float *__restrict__ bias, int act,
                                                                   float slope, int64_t act_body,
                                                                   float *__restrict__ out) {
    __shared__ float half[WT_CH][8][6][32];
    const int i = threadIdx.x / 32, lc = threadIdx.x % 32;
    const int col = blockIdx.x * 32 + lc, co0 = blockIdx.y * WT_CH;
    const int64_t stride = int64_t(g.cout) * g.cols;
    float t8[WT_CH][8];
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        const float *src = mm + int64_t(min(co0 + q, g.cout - 1)) * g.cols + col;
#pragma unroll
        for (int j = 0; j < 8; ++j) t8[q][j] = src[(i * 8 + j) * stride];
    }
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        float o[6];
        at_pass(t8[q], o);
#pragma unroll
        for (int j = 0; j < 6; ++j) half[q][i][j][lc] = o[j];
    }
    __syncthreads();
    int img, tile;
    if (i >= 6 || !column_tile(g, col, img, tile)) return;
    const int ty = tile / g.tw, tx = tile - ty * g.tw;
    const int ww = tx * 6 + i;
#pragma unroll
    for (int q = 0; q < WT_CH; ++q) {
        const int co = co0 + q;
        if (co >= g.cout) return;
        float tt[8], o[6];
#pragma unroll
        for (int r = 0; r < 8; ++r) tt[r] = half[q][r][i][lc];
        at_pass(tt, o);
        const float bv = bias ? bias[co] : 0.f;
        const int64_t plane = (int64_t(img) * g.cout + co) * g.ho * g.wo;
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            const int hh = ty * 6 + r;
            if (hh < g.ho && ww < g.wo) {
                float val = o[r];
                if (bias) val = __fadd_rn(val, bv);
                const int64_t idx = plane + hh * g.wo + ww;
                out[idx] = MISH ? apply_act(val, act, slope, idx < act_body) : apply_act_basic(val, act, slope, idx < act_body);
            }
        }
    }
}

// Y of F(2,3) (winograd_algorithm.cpp:262-330), cut to the true output, + optional bias / activation.  Thread = one
// column of one output channel.
template <bool MISH>
__global__ __launch_bounds__(256) void wino23_output_transform_kernel(const float *__restrict__ mm, WinoGeom g,
                                                                     const float *__restrict__ bias, int act,
                                                                     float slope, int64_t act_body,
                                                                     float *__restrict__ out) {
    const int col = blockIdx.x * 256 + threadIdx.x, co = blockIdx.y;
    int img, tile;
    if (col >= g.cols || !column_tile(g, col, img, tile)) return;
    const int ty = tile / g.tw, tx = tile - ty * g.tw;
    const float *src = mm + int64_t(co) * g.cols + col;
    const int64_t stride = int64_t(g.cout) * g.cols;
    float m[16], a[8], o[4];
#pragma unroll
    for (int t = 0; t < 16; ++t) m[t] = src[t * stride];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a[2 * k] = m[4 * k] + m[4 * k + 1] + m[4 * k + 2];
        a[2 * k + 1] = m[4 * k + 1] - m[4 * k + 2] - m[4 * k + 3];
    }
    o[0] = a[0] + a[2] + a[4];
    o[1] = a[1] + a[3] + a[5];
    o[2] = a[2] - a[4] - a[6];
    o[3] = a[3] - a[5] - a[7];
    const float bv = bias ? bias[co] : 0.f;
    const int64_t plane = (int64_t(img) * g.cout + co) * g.ho * g.wo;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int hh = ty * 2 + r, ww = tx * 2 + i;
            if (hh < g.ho && ww < g.wo) {
                float val = o[r * 2 + i];
                if (bias) val = __fadd_rn(val, bv);
                const int64_t idx = plane + hh * g.wo + ww;
                out[idx] = MISH ? apply_act(val, act, slope, idx < act_body) : apply_act_basic(val, act, slope, idx < act_body);
            }
        }
}

int make_geom(const tsx_conv2d_geom *q, float padding_value, WinoGeom *g, int tile) {
    TSX_REQUIRE(q, "winograd: null geometry");
    TSX_REQUIRE(q->kh == 3 && q->kw == 3 && q->stride_h == 1 && q->stride_w == 1 && q->dilation_h == 1 &&
                    q->dilation_w == 1,
                "winograd: needs a 3x3 kernel with stride 1 and dilation 1");
    TSX_REQUIRE(q->n > 0 && q->c > 0 && q->h > 0 && q->w > 0 && q->cout > 0, "winograd: non-positive extent");
    TSX_REQUIRE(q->pad_top >= 0 && q->pad_bottom >= 0 && q->pad_left >= 0 && q->pad_right >= 0,
                "winograd: negative padding is not supported");
    g->n = q->n;
    g->c = q->c;
    g->h = q->h;
    g->w = q->w;
    g->cout = q->cout;
    g->ho = q->h + q->pad_top + q->pad_bottom - 2;
    g->wo = q->w + q->pad_left + q->pad_right - 2;
    TSX_REQUIRE(g->ho > 0 && g->wo > 0, "winograd: empty output %dx%d", g->ho, g->wo);
    g->pad_top = q->pad_top;
    g->pad_left = q->pad_left;
    g->th = (g->ho + tile - 1) / tile;
    g->tw = (g->wo + tile - 1) / tile;
    TSX_REQUIRE(int64_t(g->n) * g->th * g->tw < (int64_t(1) << 30), "winograd: too many tiles");
    g->tiles = g->th * g->tw;
    g->padding_value = padding_value;
    g->rfrags = (q->cout + 31) / 32;
    g->kgroups = (q->c + 7) / 8;
    g->n8 = g->tiles / 8 * 8;
    g->mfrags = int(ceil_div(int64_t(g->n) * g->n8, 32));
    g->nfrags = g->mfrags + int(ceil_div(int64_t(g->n) * (g->tiles - g->n8), 32));
    g->cols = 32 * g->nfrags;
    return 0;
}

size_t kernel_bytes(int cout, int cin, int freqs) {
    if (cout <= 0 || cin <= 0) return 0;
    return size_t(freqs) * size_t(round_up(cout, 32)) * size_t(round_up(cin, 8)) * sizeof(float);
}

size_t operand_floats(const WinoGeom &g, int freqs) { return size_t(freqs) * g.nfrags * g.kgroups * 256; }     // V

size_t workspace_bytes(const tsx_conv2d_geom *q, int tile) {
    WinoGeom g;
    if (make_geom(q, 0.f, &g, tile)) return 0;
    const int freqs = (tile + 2) * (tile + 2);
    return (operand_floats(g, freqs) + size_t(freqs) * g.cout * g.cols) * sizeof(float);
}

template <int TILE>
int transform_kernel(int cout, int cin, const float *w, float *u, hipStream_t stream) {
    TSX_REQUIRE(cout > 0 && cin > 0 && w && u, "winograd transform_kernel: bad argument");
    const int rfrags = (cout + 31) / 32, kgroups = (cin + 7) / 8;
    hipLaunchKernelGGL(wino_kernel_transform_kernel<TILE>, dim3(unsigned(rfrags) * unsigned(kgroups)), dim3(256), 0, stream, w, cout, cin, rfrags,
                       kgroups, u);
    TSX_LAUNCH_CHECK("wino_kernel_transform_kernel");
    return 0;
}

template <int TILE>
int conv2d(const tsx_conv2d_geom *q, const float *x, const float *u, float padding_value, const float *bias, int act, float slope,
           float *out, void *workspace, size_t bytes, hipStream_t stream) {
    WinoGeom g;
    if (int rc = make_geom(q, padding_value, &g, TILE)) return rc;
    TSX_REQUIRE(x && u && out, "winograd: null argument");
    TSX_REQUIRE(act >= TSX_ACT_NONE && act <= TSX_ACT_MISH_FAST, "winograd: unknown activation %d", act);
    constexpr int FREQS = (TILE + 2) * (TILE + 2);
    const size_t need = workspace_bytes(q, TILE);
    if (!workspace || bytes < need) return fail(TSX_E_WORKSPACE, "winograd: workspace %zu < %zu bytes", bytes, need);
    TSX_REQUIRE(g.cout <= 65535 * WT_CH && g.kgroups <= 32767, "winograd: too many channels");
    float *v = static_cast<float *>(workspace), *m = v + operand_floats(g, FREQS);
    if (TILE == 6)
        hipLaunchKernelGGL(wino_input_transform_kernel, dim3(unsigned(g.nfrags), unsigned(2 * g.kgroups)), dim3(256), 0, stream, x, g, v);
    else
        hipLaunchKernelGGL(wino23_input_transform_kernel, dim3(unsigned(g.nfrags), unsigned(ceil_div(2 * g.kgroups, 8))), dim3(256), 0, stream, x,
                           g, v);
    TSX_LAUNCH_CHECK("wino_input_transform_kernel");

    // Wavefronts of a workgroup: as many as there are row fragments along these, the others along columns where the grid is large
    // enough to fill the CUs with what is left.
    const int rounds = FREQS / 8, wr = g.rfrags >= 3 ? 4 : g.rfrags, row_blocks = (g.rfrags + wr - 1) / wr;
    const int64_t frag_items = int64_t(FREQS) * row_blocks * g.mfrags;
    const int wc = frag_items > 512 ? 4 / wr : 1, tails = int(ceil_div(int64_t(g.n) * (g.tiles - g.n8), 16));
    // One column fragment per wavefront: three or four wavefronts per SIMD hide one another's loads.  Where that is more than three
    // workgroups per CU and four fragments make it one, long sums go faster so: what a CU fetches halves.  (32 images
    // 14x14, 256 to 256 channels, F(6,3): 55.2 us against 47.4 with four; 4 images 56x56, 128 to 128, F(2,3): 38.3 against 47.4.)
    const bool four = frag_items > 768 * wc && g.kgroups >= 16 && int64_t(FREQS) * row_blocks * ceil_div(ceil_div(g.mfrags, 4), wc) <= 256;
    const int fn = four ? 4 : 1;
    const int col_blocks = (g.mfrags + fn - 1) / fn;
    // The tail's fragments with the column blocks: by themselves they fetch all of U again, beside these on the same CUs (8 images
    // 28x28, 256 to 256 channels, by the wavefronts' clocks: 15 us without the tail, 20 with it, 30 with it as workgroups of its own).
    // A grid that leaves CUs idle computes them there (1 image 14x14, 512 to 512, F(2,3): 25.9 us attached, 21.7).
    const int attached = tails <= col_blocks && int64_t(FREQS) * row_blocks * ceil_div(col_blocks, wc) >= 256;
    const int64_t items = int64_t(rounds) * row_blocks * (ceil_div(col_blocks, wc) + (attached ? 0 : ceil_div(tails, wc)));
    const auto gemm = four ? wino_gemm_kernel<4> : wino_gemm_kernel<1>;
    // one launch, except where its work items would be 2^32 or more
    const int64_t most = ((int64_t(1) << 24) - 1) / 8;
    for (int64_t first = 0; first < items; first += most) {
        const dim3 grid(8u * unsigned(std::min(most, items - first)));
        hipLaunchKernelGGL(gemm, grid, dim3(256), 0, stream, u, v, m, g, wr, wc, row_blocks, col_blocks, tails, attached, rounds, first);
        TSX_LAUNCH_CHECK("wino_gemm_kernel");
    }

    const int64_t body = int64_t(g.n) * g.cout * g.ho * g.wo / 4 * 4;
    const bool mish = act >= TSX_ACT_MISH;
    if (TILE == 6) {
        const dim3 grid(unsigned(g.nfrags), unsigned(ceil_div(g.cout, WT_CH)));
        if (mish) hipLaunchKernelGGL(wino_output_transform_kernel<true>, grid, dim3(256), 0, stream, m, g, bias, act, slope, body, out);
        else hipLaunchKernelGGL(wino_output_transform_kernel<false>, grid, dim3(256), 0, stream, m, g, bias, act, slope, body, out);
    } else {
        TSX_REQUIRE(g.cout <= 65535, "winograd: too many output channels");
        const dim3 grid(unsigned(ceil_div(g.cols, 256)), unsigned(g.cout));
        if (mish) hipLaunchKernelGGL(wino23_output_transform_kernel<true>, grid, dim3(256), 0, stream, m, g, bias, act, slope, body, out);
        else hipLaunchKernelGGL(wino23_output_transform_kernel<false>, grid, dim3(256), 0, stream, m, g, bias, act, slope, body, out);
    }
    TSX_LAUNCH_CHECK("wino_output_transform_kernel");
    return 0;
}

}  // namespace
}  // namespace tsx

extern "C" {

size_t tsx_winograd_f63_kernel_bytes(int32_t cout, int32_t cin) { return tsx::kernel_bytes(cout, cin, 64); }

int tsx_winograd_f63_transform_kernel(int32_t cout, int32_t cin, const float *w_oihw_dev, float *u_dev, void *stream) {
    return tsx::transform_kernel<6>(cout, cin, w_oihw_dev, u_dev, tsx::as_stream(stream));
}

size_t tsx_winograd_f63_workspace_bytes(const tsx_conv2d_geom *q) { return tsx::workspace_bytes(q, 6); }

int tsx_conv2d_winograd_f63_nchw(const tsx_conv2d_geom *q, const float *x_dev, const float *u_dev, float padding_value,
                                 const float *bias_dev, int32_t act, float slope, float *out_dev, void *workspace_dev,
                                 size_t workspace_bytes, void *stream_) {
    return tsx::conv2d<6>(q, x_dev, u_dev, padding_value, bias_dev, act, slope, out_dev, workspace_dev, workspace_bytes, tsx::as_stream(stream_));
}

// The tolerance-based entry: the exact form is the fastest there is.
size_t tsx_winograd_f63_fast_workspace_bytes(const tsx_conv2d_geom *q) { return tsx::workspace_bytes(q, 6); }

int tsx_conv2d_winograd_f63_fast_nchw(const tsx_conv2d_geom *q, const float *x_dev, const float *u_dev, float padding_value,
                                      const float *bias_dev, int32_t act, float slope, float *out_dev, void *workspace_dev,
                                      size_t workspace_bytes, void *stream_) {
    return tsx::conv2d<6>(q, x_dev, u_dev, padding_value, bias_dev, act, slope, out_dev, workspace_dev, workspace_bytes, tsx::as_stream(stream_));
}

size_t tsx_winograd_f23_kernel_bytes(int32_t cout, int32_t cin) { return tsx::kernel_bytes(cout, cin, 16); }

int tsx_winograd_f23_transform_kernel(int32_t cout, int32_t cin, const float *w_oihw_dev, float *u_dev, void *stream) {
    return tsx::transform_kernel<2>(cout, cin, w_oihw_dev, u_dev, tsx::as_stream(stream));
}

size_t tsx_winograd_f23_workspace_bytes(const tsx_conv2d_geom *q) { return tsx::workspace_bytes(q, 2); }

int tsx_conv2d_winograd_f23_nchw(const tsx_conv2d_geom *q, const float *x_dev, const float *u_dev, float padding_value,
                                 const float *bias_dev, int32_t act, float slope, float *out_dev, void *workspace_dev,
                                 size_t workspace_bytes, void *stream_) {
    return tsx::conv2d<2>(q, x_dev, u_dev, padding_value, bias_dev, act, slope, out_dev, workspace_dev, workspace_bytes, tsx::as_stream(stream_));
}

}  // extern "C"
