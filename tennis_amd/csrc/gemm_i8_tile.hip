// int8 GEMM with many rows and columns: 8 wavefronts on a tile of 64 FR rows x 128 FC output columns.
//
// Bound: the int8 MFMA.  A wavefront owns 32 FR rows x 32 FC columns, so per K of 32 it reads FR activation operands from
// LDS and FC weight operands from global memory for FR FC MFMAs.  Per K of 64 and with FR = 4, FC = 2 the CU spends
// 1024 cycles on MFMAs, 640 on LDS (64 KiB read, 16 KiB written at 128 bytes a cycle) and 768 on the vector memory path
// (32 KiB of weights, 16 KiB of activations at 64 bytes a cycle); with weights through LDS as well that one would be full,
// and with half the fragments per wavefront the memory path would be.
//   * activations: chunks of 128 K bytes per row (whole cache lines), global -> registers -> LDS, double-buffered; the
//     16-byte pieces of a row are XORed with bits 1..3 of the row, so 16 rows cover the 256 bytes of banks for one piece (no
//     conflicts counted; with bits 0..2, which leave half the banks idle, two fifths of the LDS cycles were conflicts);
//   * weights: the packed operands are 1 KiB contiguous per fragment and half K-step and go straight into registers, a
//     chunk ahead of their MFMAs;
//   * one barrier per chunk, ahead of the chunk's last MFMAs, whose time covers the first LDS reads behind it.
// 4096 x 4096 x 4096: 67 .. 74 us with fp32 output on rounded normal operands (86 .. 105 on the window-stationary kernel's
// GEMM form; uniformly random bytes, which toggle most and get the lowest clocks: 82 us), 66 us with int8 output (155).
// Counted at this size MFMAs are busy half of a CU's time; the rest goes to operand waits around the barrier and to the
// stores, which begin everywhere when the last MFMA is done.  fp32 accumulators go out as 4-byte stores with lanes along
// columns: two whole 128-byte lines per instruction.
// int32 accumulation is exact, so the results are the other GEMM kernels' and the oracle's.
#include "gemm_i8_tile.hpp"

namespace tsx {
namespace {

constexpr int THREADS = 512;
constexpr int CHUNK = 128;             // K bytes of a row per chunk: two K-steps of 64
constexpr int HALVES = CHUNK / 32;     // MFMA steps per chunk

typedef float v4f __attribute__((ext_vector_type(4)));

// The activation over a run of values behind one uniform branch: unrolled over a wavefront's 128 values, a branch per value
// puts the taken paths an instruction-cache miss apart (4096 x 4096 fp32 outputs: 36 us of epilogue).
template <int N, class Body>
__device__ __forceinline__ void activate(float (&v)[N], const EpiParams &p, Body &&in_body) {
    if (p.act == TSX_ACT_RELU) {
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = apply_act_basic(v[r], TSX_ACT_RELU, 0.f, in_body(rc)); });
    } else if (p.act == TSX_ACT_LEAKY_RELU) {
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = apply_act_basic(v[r], TSX_ACT_LEAKY_RELU, p.slope, in_body(rc)); });
    } else if (p.act == TSX_ACT_MISH_FAST) {
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = mish_short_behind_a_branch(v[r]); });
    }
}

// COLS: MFMA columns are output columns (any epilogue); otherwise they are rows, for packed int8 output alone.
template <int FR, int FC, bool COLS>
__global__ __launch_bounds__(THREADS) void gemm_i8_tile_kernel(GemmTileParams p) {
    constexpr int ROWS = 64 * FR;
    __shared__ __attribute__((aligned(16))) int8_t lds[2][ROWS * CHUNK];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wave_r = wave >> 2, wave_c = wave & 3;
    // blockIdx % 8 is the XCD: each takes a run of consecutive tiles, which walk four row tiles before the next column
    // tile, so the runs of an XCD share rows and columns in its L2
    const int tiles = p.row_tiles * p.col_tiles;
    const int t = int(blockIdx.x % 8) * p.tiles_per_xcd + int(blockIdx.x / 8);
    if (int(blockIdx.x / 8) >= p.tiles_per_xcd || t >= tiles) return;      // uniform, ahead of every barrier
    const int group = t / (4 * p.col_tiles), in_group = t - group * 4 * p.col_tiles;
    const int group_rows = min(4, p.row_tiles - 4 * group);
    const int tile_c = in_group / group_rows, tile_r = 4 * group + in_group - tile_c * group_rows;
    const int row0 = tile_r * ROWS, frag0 = (tile_c * 4 + wave_c) * FC;
    const int frags = p.coutp / 32;
    const int chunks = (p.cblocks + 1) / 2;

    // chunk copy: thread -> piece tid % 8 of rows tid / 8 + 64 i (rows beyond m: the last one, never stored).  Scalar base
    // and 32-bit lane offsets: no address arithmetic between the MFMAs.
    const int piece = tid % 8;
    const int8_t *const x_base = p.xs + int64_t(row0) * p.pitch;
    unsigned src[FR];
    int dst[FR];
    static_for<0, FR>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int r = tid / 8 + 64 * i;
        src[i] = unsigned(min(r, p.m - 1 - row0)) * unsigned(p.pitch) + piece * 16 + 16;
        dst[i] = r * CHUNK + ((piece ^ ((r >> 1) & 7)) * 16);
    });
    // the tile of the last row, or the one before where rows are shorter than a K-step, in the last chunk: pieces must end
    // with the matrix.  Offsets carry 16 so that the limit, 15 bytes ahead of the chunk at most, is no negative one.
    const bool last_rows = int64_t(p.m - row0 - ROWS) * p.pitch < 64 && p.pitch != p.cp;
    const int limit = last_rows ? int(int64_t(p.m - row0) * p.pitch) - (chunks - 1) * CHUNK : 0;
    v4i stage[FR];
    auto stage_load = [&](int c) __attribute__((always_inline)) {
        // an odd number of K-steps ends in half a chunk: the last half again, against weights that are zero
        const int back = c * CHUNK + piece * 16 < p.cp ? 0 : 64;
        const bool clamp = last_rows && c == chunks - 1;
        static_for<0, FR>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            int off = int(src[i]) - back;
            if (clamp) off = min(off, limit);
            unsigned uoff = unsigned(off);
            asm volatile("" : "+v"(uoff));       // keeps the widening at the load, which then takes the scalar base
            stage[i] = load_piece(x_base + (c * CHUNK - 16) + uoff);
        });
    };
    auto stage_store = [&](int buf, int c) __attribute__((always_inline)) {
        if (last_rows && c == chunks - 1) {
            const int back = c * CHUNK + piece * 16 < p.cp ? 0 : 64;
            static_for<0, FR>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                stage[i] = shift_piece(stage[i], max(int(src[i]) - back - limit, 0));
            });
        }
        static_for<0, FR>([&](auto ic) { *reinterpret_cast<v4i *>(&lds[buf][dst[decltype(ic)::value]]) = stage[decltype(ic)::value]; });
    };

    // weights: packed[K-step][fragment][half][lane][16]; fragments beyond the packed columns: the last one, never stored.
    // The packed K-steps are a multiple of four, so a whole last chunk is there to be read.
    unsigned w_off[FC];
    static_for<0, FC>([&](auto fc) { w_off[decltype(fc)::value] = unsigned(min(frag0 + decltype(fc)::value, frags - 1)) * 2048u + lane * 16; });
    const int64_t w_kstride = int64_t(frags) * 2048;
    v4i w[HALVES][FC];
    auto w_load = [&](auto hc, int c) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        const int8_t *base = p.wp + (2 * c + h / 2) * w_kstride + (h % 2) * 1024;
        static_for<0, FC>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            unsigned off = w_off[f];
            asm volatile("" : "+v"(off));
            w[h][f] = *reinterpret_cast<const v4i *>(base + off);
        });
    };

    // activation operands: lane l supplies row l % 32, K bytes 16 (l / 32) .. of the half
    const int b_row = (wave_r * 32 * FR + lane % 32) * CHUNK, b_key = (lane >> 1) & 7;
    v4i b[2][FR];
    auto b_read = [&](auto sc, auto hc, int buf) __attribute__((always_inline)) {
        const int8_t *at = &lds[buf][b_row + ((2 * decltype(hc)::value + lane / 32) ^ b_key) * 16];
        static_for<0, FR>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            b[decltype(sc)::value][i] = *reinterpret_cast<const v4i *>(at + i * 32 * CHUNK);
        });
    };

    v16i acc[FR][FC];
    static_for<0, FR * FC>([&](auto fc) {
        constexpr int f = decltype(fc)::value;
        static_for<0, 16>([&](auto rc) { acc[f / FC][f % FC][decltype(rc)::value] = 0; });
    });

    stage_load(0);
    static_for<0, HALVES>([&](auto hc) { w_load(hc, 0); });
    stage_store(0, 0);
    __syncthreads();
    b_read(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, 0);
    for (int c = 0; c < chunks; ++c) {
        const int buf = c & 1;
        const int next = c + 1 < chunks ? c + 1 : c;            // behind the last chunk: its own again, never used
        stage_load(next);
        static_for<0, HALVES>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            if constexpr (h + 1 < HALVES) {
                b_read(std::integral_constant<int, (h + 1) % 2>{}, std::integral_constant<int, h + 1>{}, buf);
            } else {
                // every wavefront has its reads of this buffer's last half behind it, and those of the other buffer since
                // the barrier before: the other buffer is free, and full behind this barrier
                stage_store(buf ^ 1, next);
                __syncthreads();
                b_read(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, buf ^ 1);
            }
            // left to itself the compiler gathers the weight loads at the end of the chunk and puts every LDS read right
            // in front of its MFMA
            __builtin_amdgcn_sched_barrier(0);
            // the wavefront that has its operands goes ahead of the other one's loads (4096^3 with int8 output: 69 -> 66 us,
            // 3000^3 64 -> 54)
            __builtin_amdgcn_s_setprio(1);
            static_for<0, FR * FC>([&](auto fc) {
                constexpr int i = decltype(fc)::value / FC, f = decltype(fc)::value % FC;
                if constexpr (COLS) acc[i][f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[h % 2][i], w[h][f], acc[i][f], 0, 0, 0);
                else acc[i][f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[h][f], b[h % 2][i], acc[i][f], 0, 0, 0);
            });
            __builtin_amdgcn_s_setprio(0);
            w_load(hc, next);
            __builtin_amdgcn_sched_barrier(0);
        });
    }

    if constexpr (COLS) {
        // accumulator r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4 of the fragment, column l % 32: a store instruction
        // writes two runs of 32 consecutive columns
        const int64_t out0 = int64_t(row0) * p.cout;
        // from this element of the tile on the activation's scalar tail: the tensor's last one to three elements, which are
        // elements of several rows where there is one column
        const unsigned body = unsigned(min(max(p.act_body - out0, int64_t(0)), int64_t(0xffffffff)));
        int co[FC];
        float dq[FC], bias[FC];
        static_for<0, FC>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            co[f] = (frag0 + f) * 32 + lane % 32;
            const bool in = co[f] < p.cout;
            dq[f] = (in && p.dq) ? p.dq[co[f]] : 0.f;
            bias[f] = (in && p.bias) ? p.bias[co[f]] : 0.f;
        });
        static_for<0, FR>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int first = (wave_r * FR + i) * 32 + 4 * (lane / 32), rows = p.m - row0;      // rows of the tile
            float rs[16], qs[16];
            if (p.row_scale)
                static_for<0, 16>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    rs[r] = p.row_scale[row0 + min(first + 8 * (r / 4) + r % 4, rows - 1)];
                });
            if (p.out_i8)
                static_for<0, 16>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    const int row = min(first + 8 * (r / 4) + r % 4, rows - 1);
                    qs[r] = p.q_scales[row0 + row];
                });
            static_for<0, FC>([&](auto fc) {
                constexpr int f = decltype(fc)::value;
                unsigned off[16];
                static_for<0, 16>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    off[r] = unsigned(first + 8 * (r / 4) + r % 4) * unsigned(p.cout) + co[f];
                });
                auto stored = [&](auto rc) { constexpr int r = decltype(rc)::value; return first + 8 * (r / 4) + r % 4 < rows && co[f] < p.cout; };
                if (p.out_acc)
                    static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; if (stored(rc)) (p.out_acc + out0)[off[r]] = acc[i][f][r]; });
                if (p.out_f32 || p.out_i8) {
                    float v[16];
                    static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fmul_rn(float(acc[i][f][r]), dq[f]); });
                    if (p.row_scale) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fmul_rn(v[r], rs[r]); });
                    if (p.bias) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], bias[f]); });
                    activate(v, p, [&](auto rc) { constexpr int r = decltype(rc)::value; return off[r] < body; });
                    if (p.out_f32)
                        static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; if (stored(rc)) (p.out_f32 + out0)[off[r]] = v[r]; });
                    if (p.out_i8)
                        static_for<0, 16>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            if (stored(rc)) (p.out_i8 + out0)[off[r]] = int8_t(quantize_value(__fmul_rn(v[r], qs[r]), false));
                        });
                }
            });
        });
    } else {
        // accumulator r of lane l: column 8 (r / 4) + 4 (l / 32) + r % 4 of the fragment, row l % 32.  The columns are a
        // multiple of 16, so every element is in the activation's body; two half-wave swaps leave every lane with 16
        // consecutive columns -- lower half 0..15, upper half 16..31 -- for one store.
        static_for<0, FC>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            const int cf = (frag0 + f) * 32;
            if (cf < p.cout) {                                   // uniform
                v4f dq[4], bias[4];
                static_for<0, 4>([&](auto gc) {
                    constexpr int g = decltype(gc)::value;
                    const v4f z = {0.f, 0.f, 0.f, 0.f};
                    const int co = min(cf + 8 * g + 4 * (lane / 32), p.cout - 4);
                    dq[g] = *reinterpret_cast<const v4f *>(p.dq + co);
                    bias[g] = p.bias ? *reinterpret_cast<const v4f *>(p.bias + co) : z;
                });
                static_for<0, FR>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int row = row0 + (wave_r * FR + i) * 32 + lane % 32;
                    const int in_row = min(row, p.m - 1);
                    const float rs = p.row_scale ? p.row_scale[in_row] : 0.f, qs = p.q_scales[in_row];
                    uint32_t word[4];
                    float v[16];
                    static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fmul_rn(float(acc[i][f][r]), dq[r / 4][r % 4]); });
                    if (p.row_scale) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fmul_rn(v[r], rs); });
                    if (p.bias) static_for<0, 16>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], bias[r / 4][r % 4]); });
                    activate(v, p, [](auto) { return true; });
                    quantize_words(v, qs, false, word);
                    const auto s02 = __builtin_amdgcn_permlane32_swap(word[0], word[2], false, false);
                    const auto s13 = __builtin_amdgcn_permlane32_swap(word[1], word[3], false, false);
                    const int co = cf + 16 * (lane / 32);
                    const v4i packed = {int(s02[0]), int(s02[1]), int(s13[0]), int(s13[1])};
                    if (row < p.m && co < p.cout) *reinterpret_cast<v4i *>(p.out_i8 + int64_t(row) * p.cout + co) = packed;
                });
            }
        });
    }
}

template <int FR, int FC>
int launch(GemmTileParams p, hipStream_t stream) {
    p.row_tiles = int(ceil_div(p.m, 64 * FR));
    p.col_tiles = int(ceil_div(p.cout, 128 * FC));
    p.tiles_per_xcd = int(ceil_div(int64_t(p.row_tiles) * p.col_tiles, 8));
    const bool packed = p.out_i8 && !p.out_f32 && !p.out_acc && p.cout % 16 == 0 &&
                        reinterpret_cast<uintptr_t>(p.out_i8) % 16 == 0 && reinterpret_cast<uintptr_t>(p.dq) % 16 == 0 &&
                        reinterpret_cast<uintptr_t>(p.bias) % 16 == 0;
    const dim3 grid(unsigned(8 * p.tiles_per_xcd));
    if (packed) hipLaunchKernelGGL((gemm_i8_tile_kernel<FR, FC, false>), grid, dim3(THREADS), 0, stream, p);
    else hipLaunchKernelGGL((gemm_i8_tile_kernel<FR, FC, true>), grid, dim3(THREADS), 0, stream, p);
    TSX_LAUNCH_CHECK("gemm_i8_tile_kernel");
    return 0;
}

}  // namespace

int gemm_i8_tile_choose(int m, int n, int k, bool int8_out, bool unpadded) {
    // One workgroup of any tile fills a CU's issue slots, so a launch takes rounds of 256 tiles; a round takes the tile's
    // fixed part (first loads, epilogue) and a time per 128 of K, in us as fitted to the sweeps quoted below.
    static const float fixed_f32[3] = {7.f, 10.f, 16.f}, fixed_i8[3] = {5.f, 8.5f, 12.f}, per_chunk[3] = {0.57f, 0.9f, 1.75f};
    const int64_t chunks = ceil_div(k, CHUNK);
    int best = 0;
    int64_t best_tiles = 0;
    float best_cost = 0.f;
    for (int t = 1; t <= 3; ++t) {
        const int64_t tiles = ceil_div(m, t == 3 ? 256 : 128) * ceil_div(n, t == 1 ? 128 : 256);
        const float cost = float(ceil_div(tiles, 256)) * ((int8_out ? fixed_i8 : fixed_f32)[t - 1] + float(chunks) * per_chunk[t - 1]);
        if (!best || cost < best_cost) {
            best = t;
            best_tiles = tiles;
            best_cost = cost;
        }
    }
    // Against the window-stationary kernel's GEMM form.  fp32 output: that kernel's smaller tiles spread a problem of few
    // tiles over more CUs (1024 x 1024 x 1024, 64 tiles of 128 x 128: 6.7 us there, 9.6 here; 4096 x 512 columns, K = 4096,
    // 128 tiles: 20 and 24); from three quarters of a round on this one is ahead (2048^3: 19.5 and 17.7; 2048 x 4096, K =
    // 4096: 48 and 42; 4096^3: 92 .. 105 and 75.6; 1500 x 3000, K = 700, 144 tiles of 128 x 256: 22.6 and 19.3).
    // int8 output: that kernel divides by the row length for each element, so packed stores win everywhere (512^3: 11.6
    // and 5.8; 256 x 1024 x 1024: 12.9 and 7.4; 4096^3: 155 and 69); single bytes, where the columns are no multiple of
    // 16, only from half a round on (777 x 1111, K = 1500, 63 tiles: 19.1 and 19.9; 3000^3: 92 and 65).
    // Rows that the other kernel would need copied first: always (732 x 226, K = 177, with the copy 17, here 8 us).
    if (unpadded) return best;
    if (int8_out) return n % 16 == 0 || best_tiles >= 128 ? best : 0;
    return best_tiles >= (best == 1 ? 192 : 144) ? best : 0;
}

int gemm_i8_tile_launch(const GemmTileParams &p, int tile, hipStream_t stream) {
    return tile == 3 ? launch<4, 2>(p, stream) : tile == 2 ? launch<2, 2>(p, stream) : launch<2, 1>(p, stream);
}

}  // namespace tsx
