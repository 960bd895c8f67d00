// fp32 convolution on v_mfma_f32_32x32x2_f32 for layers with more than a few hundred 32 x 32 output tiles (cpu::Conv2DCore,
// src/kernels/cpu/conv2d_core.cpp:17-119) and the plain matrix product of inner_prod (src/kernels/cpu/inner_prod.cpp:19-74),
// which is a 1x1 convolution over one image of one row.
//
// The fp32 matrix cores need 64 cycles per instruction, so an operand costs little to read and the kernel is bound by
// them as long as nothing else gets in the way.  What got in the way of the im2col form (gemm_f32.hip: 205 us on 8 images
// of 28x28x256 with 256 3x3 filters, 36 TFLOP/s) is the gather: nine loads, address computations and bounds tests per
// input element.  Here K is walked in chunks of `cc` input channels; a chunk's input PATCH -- the rows and columns that
// the tile's positions read through all taps, padding included as values -- is copied to LDS once per element, and
// every tap is a shifted read of it: the MFMA step (channel pair, tap) takes channel 2p for lanes 0..31 and 2p + 1 for
// lanes 32..63, position l%32 each.  Where a thread's patch elements lie is computed once; from chunk to chunk only a
// uniform base moves.  The chunk's weights go to LDS transposed, [channel x tap][row], read without conflicts.  The next
// chunk's loads are in flight during the MFMAs; two or more workgroups per CU cover each other's barriers.
//
// Tiles of BM = 32 WM FM output channels x BN = 32 WN FN positions, 4 wavefronts as WM x WN x WK; with WK > 1 the
// wavefronts split a chunk's channel pairs and add their partial tiles through LDS in a fixed order.  Positions are
// numbered over the whole batch ("flat": a tile may cross rows and images), or, on maps so wide that a flat tile's
// whole-row patch would hold many times its positions, a fragment is 32 columns of one row and a tile BN/32 rows of
// them ("segments").
#include "gemm_f32.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>

namespace tsx {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int WIN_THREADS = 256;

// Channels per chunk of a 1x1 instantiation (the others take 8, 4 or 2 by their patch: 8 slots of 256 elements).
constexpr int win_point_channels(int frags_per_wave) { return frags_per_wave == 1 ? 64 : 32; }
// What a thread copies per chunk: patch elements (groups of 4 of them: BV) and weights (pieces of 4: AV).  All of it
// is loaded and stored without a branch -- what is no item reads nothing (a buffer load beyond the bounds) and goes to
// LDS nothing reads -- because a load behind a branch is waited for before the next one is issued.
constexpr int win_patch_slots(int taps, int cc, int bn, bool bv) { return taps != 1 ? 8 : bv ? bn * cc / 1024 : bn * cc / 256; }
constexpr int win_weight_slots(int taps, int cc, int bm, bool av) { return av ? bm / 32 * ((cc * taps + 31) / 32) : taps == 1 ? bm * cc / 256 : 16; }
// LDS in floats, per chunk buffer: the chunk's weights and room behind them for the pieces that are none, then the patch.
constexpr int win_patch_start(int kc, int bm) { return ((kc + 4) * (bm + 1) + 3) / 4 * 4; }
constexpr int win_buffer_floats(int taps, int cc, int kc, int bm, int bn, bool bv) {
    return win_patch_start(kc, bm) + WIN_THREADS * win_patch_slots(taps, cc, bn, bv) * (bv ? 4 : 1);
}

struct WinParams {
    const float *x, *w, *bias;
    float *out;
    int M, N, K;                   // output channels, positions (n ho wo), c kh kw
    int n, C, H, W, kh, kw, dil_h, dil_w, sh, sw, pad_top, pad_left;
    int ho, wo, howo;
    int hv;                        // rows of one image with the padding its windows reach
    int wv;                        // patch columns
    int seg, col_tiles;            // segments: column tiles per row
    int cc, tiles_m, tiles_n;
    float padding_value;
    int act;
    float slope;
    int64_t act_body;
};

// TAPS: 9 (3x3 without column dilation), 1 (1x1: the patch is the tile's positions themselves, at any stride), 0 (any
// kernel).  CC: channels per chunk.  AV: weights read 4 at a time (K a multiple of 4, 16-byte aligned).  BV: 1x1 stride 1
// without padding on maps of a multiple of 4 positions: the patch is read 4 positions at a time.
// fp32 MFMAs and vector instructions share their execution units (an address addition per operand read cost 20 % of the
// kernel), so the unrolled steps hold none: a thread's global and LDS addresses are a few registers, everything else is
// uniform or an immediate -- a channel of the patch has a fixed pitch, and the code of the two buffers is separate.
template <int WM, int WN, int WK, int FM, int FN, int TAPS, int CC, bool AV, bool BV>
__global__ __launch_bounds__(WIN_THREADS) void conv_f32_window_kernel(WinParams p) {
    static_assert(WM * WN * WK == 4 && (TAPS == 1 || !BV) && (TAPS != 0 || !AV) && (TAPS == 0 || CC / 2 % WK == 0),
                  "four wavefronts; vector patches are 1x1; every wavefront has steps");
    constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN, RP = BM + 1;
    constexpr int NA = win_weight_slots(TAPS, CC, BM, AV), NB = win_patch_slots(TAPS, CC, BN, BV);
    constexpr int SPC = TAPS != 1 ? 8 / CC : 1;            // 256-element slots per channel of a patch
    constexpr int PITCH = TAPS != 1 ? 256 * SPC : BN;      // LDS floats per channel of it
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int hf = lane / 32;
    const int wk = wave % WK, wn = (wave / WK) % WN, wm = wave / (WK * WN);
    const int taps = TAPS ? TAPS : p.kh * p.kw;

    // Tiles that share their positions are consecutive, and each XCD takes a contiguous run of tiles: a patch is fetched
    // into one L2.
    const int total = p.tiles_m * p.tiles_n, per_xcd = (total + 7) / 8;
    const int t = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
    if (int(blockIdx.x >> 3) >= per_xcd || t >= total) return;
    const int tn = t / p.tiles_m, m0 = (t - tn * p.tiles_m) * BM;

    // ---- positions
    // segments: image, first row inside it, first column
    const int seg_rows = (p.ho + BN / 32 - 1) / (BN / 32), seg_tile = p.seg ? tn / p.col_tiles : 0, seg_img = seg_tile / seg_rows;
    const int seg_row = (seg_tile - seg_img * seg_rows) * (BN / 32);
    const int col0 = p.seg ? (tn - seg_tile * p.col_tiles) * 32 : 0;
    auto decode = [&](int q, int &row, int &col) -> bool {                 // tile position -> batch-wide output row, column
        if (p.seg) {
            row = seg_img * p.ho + seg_row + q / 32;
            col = col0 + q % 32;
            return seg_row + q / 32 < p.ho && col < p.wo;
        }
        const int pos = tn * BN + q;
        row = pos / p.wo;
        col = pos - row * p.wo;
        return pos < p.N;
    };
    auto virtual_row = [&](int row) { const int img = row / p.ho; return img * p.hv + (row - img * p.ho) * p.sh; };
    const int first_row = p.seg ? seg_img * p.ho + seg_row : tn * BN / p.wo;
    const int vr0 = virtual_row(first_row);
    const int kc = CC * taps;                                              // K of a chunk
    const int patch_start = win_patch_start(kc, BM), buffer = win_buffer_floats(TAPS, CC, kc, BM, BN, BV);

    // ---- patch bookkeeping.  Slot i of a thread is element tid + 256 (i % SPC) of channel i / SPC; 1x1: always the same
    // position(s), of channel tid / positions + i rounds.  One byte offset per element, the channel is a scalar offset.
    constexpr unsigned NOWHERE = 0x80000000u;                              // beyond any buffer: loads 0, reads nothing
    const unsigned plane = unsigned(p.H) * unsigned(p.W);
    constexpr int ROUND = BV ? 4 * WIN_THREADS / BN : WIN_THREADS / BN;    // 1x1: channels a slot covers
    unsigned b_off[SPC], b_pad = 0;                                        // bit: the element is padding
    static_for<0, SPC>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        bool in;
        unsigned off;
        if (TAPS == 1) {
            constexpr int PER = BV ? BN / 4 : BN;
            const int pos = tn * BN + (tid % PER) * (BV ? 4 : 1);
            const int img = pos / p.howo, r = pos - img * p.howo;
            int h = 0, w = r;
            if (!BV) {
                const int oh = r / p.wo;
                h = oh * p.sh - p.pad_top;
                w = (r - oh * p.wo) * p.sw - p.pad_left;
            }
            in = pos < p.N && tid / PER < p.C && (BV || (h >= 0 && h < p.H && w >= 0 && w < p.W));
            off = (unsigned(img) * unsigned(p.C) + unsigned(tid / PER)) * plane + unsigned(h * p.W + w);
        } else {
            const int e = tid + 256 * i;
            const int pr = e / p.wv, v = vr0 + pr, img = v / p.hv;
            const int h = v - img * p.hv - p.pad_top, w = e - pr * p.wv + col0 * p.sw - p.pad_left;
            in = img < p.n && h >= 0 && h < p.H && w >= 0 && w < p.W;      // elements behind the tile's patch: loaded, never used
            off = unsigned(img) * unsigned(p.C) * plane + unsigned(h * p.W + w);
        }
        b_pad |= unsigned(!in) << i;
        b_off[i] = in ? off * 4u : NOWHERE;
    });
    // ---- weight bookkeeping.  Vector form: a wavefront copies 8 rows x 8 pieces of 4 at a time (whole cache lines in,
    // stores to LDS two to a bank), slot i = rows 8 wave + 32 (i % (BM/32)), pieces 8 (i / (BM/32)): one register per
    // row group, one LDS index, and a second set for the last pieces, of which not all exist.  Scalar form: consecutive threads
    // along K.  Rows beyond M load 0 or another row's weights; they are never stored to the output.
    constexpr int RG = BM / 32, KG = AV ? NA / RG : 1;                     // row and piece groups of a wavefront
    unsigned a_off[AV ? RG : NA], a_off_last[RG];
    int a_dst[AV ? 1 : NA], a_dst_last = 0;
    if constexpr (AV) {
        const bool piece = 32 * (KG - 1) + 4 * (lane % 8) < kc;
        static_for<0, RG>([&](auto gc) {
            constexpr int g = decltype(gc)::value;
            const int row = m0 + 32 * g + 8 * wave + lane / 8;
            a_off[g] = row < p.M ? (unsigned(row) * unsigned(p.K) + unsigned(4 * (lane % 8))) * 4u : NOWHERE;
            a_off_last[g] = piece ? a_off[g] : NOWHERE;
        });
        a_dst[0] = 4 * (lane % 8) * RP + 8 * wave + lane / 8;
        a_dst_last = piece ? a_dst[0] : (kc - 32 * (KG - 1)) * RP;         // the room behind the weights
    } else {
        static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int item = tid + i * WIN_THREADS;
            const int row = item / kc, kk = item - row * kc;
            a_off[i] = row < BM ? (unsigned(min(m0 + row, p.M - 1)) * unsigned(p.K) + unsigned(kk)) * 4u : NOWHERE;
            a_dst[i] = row < BM ? kk * RP + row : kc * RP;
        });
    }

    float b_reg[NB][BV ? 4 : 1], a_reg[NA][AV ? 4 : 1];
    const int x_bytes = int(int64_t(p.n) * p.C * plane * 4), w_bytes = int(int64_t(p.M) * p.K * 4);      // below 2 GiB
    auto load_chunk = [&](int c0) __attribute__((always_inline)) {
        const int x_at = c0 * int(plane) * 4, w_at = c0 * taps * 4;
        const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(p.x) + x_at), 0, x_bytes - x_at, 0x00020000);
        const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(p.w) + w_at), 0, w_bytes - w_at, 0x00020000);
        static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (AV) {
                const unsigned off = (i / RG == KG - 1 ? a_off_last[i % RG] : a_off[i % RG]) + 128u * (i / RG);
                const v4f q = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(wr, int(off), 0, 0));
                static_for<0, 4>([&](auto jc) { a_reg[i][decltype(jc)::value] = q[decltype(jc)::value]; });
            } else {
                a_reg[i][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wr, int(a_off[i]), 0, 0));
            }
        });
        static_for<0, NB>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            // A slot beyond the last channel reads the last one's data (zeroed in finish_chunk), never memory behind the
            // tensor.  1x1: a slot covers several channels, some of which may lie beyond: there the whole offset is what
            // is checked against the buffer's bounds.
            const int so = min(TAPS == 1 ? i * ROUND : i / SPC, p.C - 1 - c0) * int(plane) * 4;
            const int vo = int(b_off[i % SPC]) + (TAPS == 1 ? so : 0);
            if constexpr (BV) {
                const v4f q = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(xr, vo, 0, 0));
                static_for<0, 4>([&](auto jc) { b_reg[i][decltype(jc)::value] = q[decltype(jc)::value]; });
            } else {
                b_reg[i][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, vo, TAPS == 1 ? 0 : so, 0));
            }
        });
    };
    // What has arrived for chunk c0, made ready for LDS: padding elements (they have loaded 0), and zeros behind the last
    // channel of a layer whose channels end inside the chunk.
    auto finish_chunk = [&](int c0) __attribute__((always_inline)) {
        if (!BV && p.padding_value != 0.f) {
            static_for<0, NB>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                b_reg[i][0] = (b_pad >> (i % SPC)) & 1u ? p.padding_value : b_reg[i][0];
            });
        }
        if (c0 + CC > p.C) {
            const int left = p.C - c0, k_left = left * taps;
            static_for<0, NA>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                // AV: K and the piece's k are multiples of 4, it is in or out
                const bool live = AV ? 32 * (i / RG) + 4 * (lane % 8) < k_left : a_dst[AV ? 0 : i] / RP < k_left;
                static_for<0, AV ? 4 : 1>([&](auto jc) { a_reg[i][decltype(jc)::value] = live ? a_reg[i][decltype(jc)::value] : 0.f; });
            });
            static_for<0, NB>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const bool live = (TAPS == 1 ? tid / (BV ? BN / 4 : BN) + i * ROUND : i / SPC) < left;
                static_for<0, BV ? 4 : 1>([&](auto jc) { b_reg[i][decltype(jc)::value] = live ? b_reg[i][decltype(jc)::value] : 0.f; });
            });
        }
    };
    auto store_weight = [&](auto ic, int at) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        const int dst = !AV ? a_dst[AV ? 0 : i] : i / RG == KG - 1 ? a_dst_last : a_dst[0];
        static_for<0, AV ? 4 : 1>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            lds[dst + at + (AV ? 32 * (i % RG) + (32 * (i / RG) + j) * RP : 0)] = a_reg[i][j];
        });
    };
    auto store_patch = [&](auto ic, int at) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (BV) *reinterpret_cast<v4f *>(lds + tid * 4 + at + patch_start + i * WIN_THREADS * 4) = v4f{b_reg[i][0], b_reg[i][1], b_reg[i][2], b_reg[i][3]};
        else lds[tid + at + patch_start + i * WIN_THREADS] = b_reg[i][0];
    };

    // ---- this lane's positions in the patch, one LDS index per kernel row
    constexpr int KR = TAPS == 9 ? 3 : 1;
    int b_at[FN][KR];
    static_for<0, FN>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const int q = (wn * FN + j) * 32 + lane % 32;
        int row, col;
        const bool ok = decode(q, row, col);
        const int cell = TAPS == 1 ? q : ok ? (virtual_row(row) - vr0) * p.wv + (col - col0) * p.sw : 0;
        static_for<0, KR>([&](auto rc) {
            b_at[j][decltype(rc)::value] = patch_start + (hf + 2 * wk) * PITCH + cell + decltype(rc)::value * p.dil_h * p.wv;
        });
    });
    const int a_at = wm * FM * 32 + lane % 32 + (hf + 2 * wk) * taps * RP;
    v16f acc[FM][FN];
    static_for<0, FM * FN>([&](auto fc) {
        static_for<0, 16>([&](auto rc) { acc[decltype(fc)::value / FN][decltype(fc)::value % FN][decltype(rc)::value] = 0.f; });
    });

    // ---- the first chunk, and the second one's loads
    load_chunk(0);
    finish_chunk(0);
    static_for<0, NA>([&](auto ic) { store_weight(ic, 0); });
    static_for<0, NB>([&](auto ic) { store_patch(ic, 0); });
    const int last = (p.C - 1) / CC * CC;      // the last chunk; beyond it its data again, never used
    load_chunk(min(CC, last));
    __syncthreads();

    // The steps of the chunk in buffer `nowc` while the next chunk goes into the other one.  Operands are read AHEAD steps
    // before their MFMAs, across chunks as well: once the last reads of this buffer have returned and the other one is
    // stored -- the barrier -- the first reads of the next chunk run under the last MFMAs of this one.  Under the first steps
    // the next chunk's data goes to LDS, then the chunk behind it is requested.  The scheduler is held to that order (left
    // alone it gathers the reads in front of their uses and waits for them).
    if constexpr (TAPS != 0) {
        constexpr int STEPS = CC / 2 / WK * TAPS, AHEAD = STEPS % 6 == 0 ? 6 : STEPS == 9 ? 3 : 4;
        static_assert(STEPS % AHEAD == 0 && STEPS >= 2 * AHEAD, "a step's operand slot is its number modulo the ring");
        constexpr int STORES = NA + NB, PER = (STORES + STEPS / 4 - 1) / (STEPS / 4);
        float a[AHEAD][FM], b[AHEAD][FN];
        auto read = [&](auto sc, int at) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value, slot = s % AHEAD, pair = s / TAPS, tap = s % TAPS;
            static_for<0, FM>([&](auto ic) { a[slot][decltype(ic)::value] = lds[a_at + at + (2 * pair * WK * TAPS + tap) * RP + decltype(ic)::value * 32]; });
            static_for<0, FN>([&](auto jc) { b[slot][decltype(jc)::value] = lds[b_at[decltype(jc)::value][KR == 3 ? tap / 3 : 0] + at + 2 * pair * WK * PITCH + (KR == 3 ? tap % 3 : 0)]; });
        };
        auto chunk = [&](auto nowc, int c0) __attribute__((always_inline)) {
            const int now = decltype(nowc)::value * buffer, next = (1 - decltype(nowc)::value) * buffer;
            finish_chunk(min(c0 + CC, last));
            static_for<0, STEPS>([&](auto sc) {
                constexpr int s = decltype(sc)::value, slot = s % AHEAD;
                if constexpr (s + AHEAD == STEPS) __syncthreads();
                static_for<0, FM * FN>([&](auto fc) {
                    constexpr int i = decltype(fc)::value / FN, j = decltype(fc)::value % FN;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[slot][i], b[slot][j], acc[i][j], 0, 0, 0);
                });
                if constexpr (s + AHEAD < STEPS) read(std::integral_constant<int, s + AHEAD>{}, now);
                else read(std::integral_constant<int, s + AHEAD - STEPS>{}, next);
                static_for<s * PER, (s + 1) * PER>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    if constexpr (i < NA) store_weight(ic, next);
                    else if constexpr (i < STORES) store_patch(std::integral_constant<int, i - NA>{}, next);
                });
                if constexpr (s == (STORES + PER - 1) / PER) load_chunk(min(c0 + 2 * CC, last));
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        static_for<0, AHEAD>([&](auto sc) { read(sc, 0); });
        for (int c0 = 0;;) {
            chunk(std::integral_constant<int, 0>{}, c0);
            if ((c0 += CC) > last) break;
            chunk(std::integral_constant<int, 1>{}, c0);
            if ((c0 += CC) > last) break;
        }
        if constexpr (WK > 1) __syncthreads(); // the reads ahead have returned: the chunks' space can take partial tiles
    } else {
        for (int c0 = 0, now = 0; c0 <= last; c0 += CC, now ^= buffer) {
            const int next = now ^ buffer;
            finish_chunk(min(c0 + CC, last));
            static_for<0, NA>([&](auto ic) { store_weight(ic, next); });
            static_for<0, NB>([&](auto ic) { store_patch(ic, next); });
            load_chunk(min(c0 + 2 * CC, last));
            // (channel pair, kernel row, column) steps, walked by the read pointer AHEAD steps in front of the MFMAs
            constexpr int AHEAD = 4;
            const int steps = max(0, ((min(CC, p.C - c0) + 1) / 2 - wk + WK - 1) / WK) * taps;
            int a_i = a_at + now, b_i = now, r = 0, q = 0;
            float a[AHEAD][FM], b[AHEAD][FN];
            auto read = [&](auto sc) __attribute__((always_inline)) {
                constexpr int slot = decltype(sc)::value;
                static_for<0, FM>([&](auto ic) { a[slot][decltype(ic)::value] = lds[a_i + decltype(ic)::value * 32]; });
                static_for<0, FN>([&](auto jc) { b[slot][decltype(jc)::value] = lds[b_at[decltype(jc)::value][0] + b_i]; });
                a_i += RP;
                b_i += p.dil_w;
                if (++q == p.kw) {
                    q = 0;
                    b_i += p.dil_h * p.wv - p.kw * p.dil_w;
                    if (++r == p.kh) {
                        r = 0;
                        b_i += 2 * WK * PITCH - p.kh * p.dil_h * p.wv;
                        a_i += (2 * WK - 1) * taps * RP;
                    }
                }
            };
            static_for<0, AHEAD>([&](auto sc) { if (decltype(sc)::value < steps) read(sc); });
            for (int s = 0; s < steps; s += AHEAD)
                static_for<0, AHEAD>([&](auto sc) {
                    constexpr int slot = decltype(sc)::value;
                    if (s + slot < steps) {
                        static_for<0, FM * FN>([&](auto fc) {
                            constexpr int i = decltype(fc)::value / FN, j = decltype(fc)::value % FN;
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[slot][i], b[slot][j], acc[i][j], 0, 0, 0);
                        });
                        if (s + slot + AHEAD < steps) read(sc);
                    }
                });
            __syncthreads();                   // the other buffer is complete, this one fully consumed
        }
    }

    // ---- bias values of the tile's rows, requested together (one in the store loop would cost a memory round trip per row)
    float bias[FM][16];
    static_for<0, FM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        static_for<0, 16>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            bias[i][r] = p.bias && wk == 0 ? p.bias[min(m0 + (wm * FM + i) * 32 + 8 * (r / 4) + 4 * hf + r % 4, p.M - 1)] : 0.f;
        });
    });
    if constexpr (WK > 1) {
        constexpr int SLOT = WM * WN * FM * FN * 16 * 64;
        float *red = lds + (wm * WN + wn) * FM * FN * 16 * 64 + lane;      // the chunks' space takes the partial tiles
        if (wk > 0)
            static_for<0, FM * FN * 16>([&](auto rc) {
                constexpr int f = decltype(rc)::value / 16, r = decltype(rc)::value % 16;
                red[(wk - 1) * SLOT + (f * 16 + r) * 64] = acc[f / FN][f % FN][r];
            });
        __syncthreads();
        if (wk > 0) return;
        static_for<0, WK - 1>([&](auto sc) {
            static_for<0, FM * FN * 16>([&](auto rc) {
                constexpr int f = decltype(rc)::value / 16, r = decltype(rc)::value % 16;
                acc[f / FN][f % FN][r] += red[decltype(sc)::value * SLOT + (f * 16 + r) * 64];
            });
        });
    }
    // A lane's element of a row is its own offset plus a uniform one; 32-bit offsets, the output is below 2 GiB.
    const auto out = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, int(int64_t(p.M) * p.N * 4), 0x00020000);
    const bool body = p.act_body == int64_t(p.M) * p.N;      // no element behind the activation's SIMD body
    static_for<0, FN>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        int row, col;
        const bool ok = decode((wn * FN + j) * 32 + lane % 32, row, col);
        const int img = row / p.ho;
        const int base = img * p.M * p.howo + (row - img * p.ho) * p.wo + col + (m0 + wm * FM * 32 + 4 * hf) * p.howo;
        static_for<0, FM * 16>([&](auto rc) {
            constexpr int i = decltype(rc)::value / 16, r = decltype(rc)::value % 16, up = 32 * i + 8 * (r / 4) + r % 4;
            float v = acc[i][j][r];
            if (p.bias) v = __fadd_rn(v, bias[i][r]);
            v = apply_act_basic(v, p.act, p.slope, body || base + up * p.howo < p.act_body);
            const bool in = ok && m0 + wm * FM * 32 + 4 * hf + up < p.M;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), out, in ? base * 4 : int(NOWHERE), up * p.howo * 4, 0);
        });
    });
}

template <int WM, int WN, int WK, int FM, int FN, int TAPS, int CC, bool AV, bool BV>
int launch_window(const WinParams &p, size_t lds_bytes, hipStream_t stream) {
    auto kernel = conv_f32_window_kernel<WM, WN, WK, FM, FN, TAPS, CC, AV, BV>;
    if (lds_bytes > 65536) {                   // dynamic LDS beyond 64 KiB is granted per kernel and device
        static std::atomic<bool> granted[64];
        int dev = 0;
        TSX_HIP(hipGetDevice(&dev));
        if (dev >= 64 || !granted[dev].load()) {
            TSX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            if (dev < 64) granted[dev].store(true);
        }
    }
    const int total = p.tiles_m * p.tiles_n;
    hipLaunchKernelGGL(kernel, dim3(unsigned((total + 7) / 8 * 8)), dim3(WIN_THREADS), lds_bytes, stream, p);
    TSX_LAUNCH_CHECK("conv_f32_window_kernel");
    return 0;
}

struct WinTile {
    int wm, wn, wk, fm, fn;
    int bm() const { return 32 * wm * fm; }
    int bn() const { return 32 * wn * fn; }
};
constexpr WinTile WIN_TILES[] = {{1, 1, 4, 1, 1}, {1, 4, 1, 1, 1}, {2, 2, 1, 1, 1}, {2, 2, 1, 1, 2}, {2, 2, 1, 2, 2}};
constexpr int WIN_TILE_COUNT = int(sizeof(WIN_TILES) / sizeof(WIN_TILES[0]));

// The launch of one layer with one tile; false if the tile's patch does not fit.
bool plan_tile(const ConvF32Layer &l, int tile, bool flat, WinParams *p, size_t *lds_bytes, int *kind, bool *av, bool *bv) {
    const WinTile &t = WIN_TILES[tile];
    const int taps = l.kh * l.kw, bn = t.bn(), bm = t.bm();
    const bool point = taps == 1;
    p->M = l.cout;
    p->K = l.c * taps;
    p->N = int(int64_t(l.n) * l.ho * l.wo);
    p->n = l.n; p->C = l.c; p->H = l.h; p->W = l.w;
    p->kh = l.kh; p->kw = l.kw; p->dil_h = l.dil_h; p->dil_w = l.dil_w; p->sh = l.stride_h; p->sw = l.stride_w;
    p->pad_top = l.pad_top; p->pad_left = l.pad_left;
    p->ho = l.ho; p->wo = l.wo; p->howo = l.ho * l.wo;
    p->hv = (l.ho - 1) * l.stride_h + (l.kh - 1) * l.dil_h + 1;
    p->tiles_m = int(ceil_div(l.cout, bm));
    if (flat) {
        p->seg = 0;
        p->col_tiles = 1;
        p->wv = (l.wo - 1) * l.stride_w + (l.kw - 1) * l.dil_w + 1;
        p->tiles_n = int(ceil_div(p->N, bn));
    } else {
        p->seg = 1;
        p->col_tiles = int(ceil_div(l.wo, 32));
        p->wv = 31 * l.stride_w + (l.kw - 1) * l.dil_w + 1;
        p->tiles_n = int(int64_t(l.n) * ceil_div(l.ho, bn / 32)) * p->col_tiles;
    }
    if (int64_t(p->tiles_m) * p->tiles_n >= (int64_t(1) << 30)) return false;
    *av = p->K % 4 == 0 && reinterpret_cast<uintptr_t>(l.w_dev) % 16 == 0;
    *bv = point && l.stride_h == 1 && l.stride_w == 1 && l.pad_top == 0 && l.pad_left == 0 && p->howo % 4 == 0 && l.ho == l.h && l.wo == l.w &&
          reinterpret_cast<uintptr_t>(l.x_dev) % 16 == 0;
    int64_t cells = bn;
    if (!point) {
        // rows of the largest patch: output rows a tile touches, and per image border it crosses the padding rows between
        const int64_t rows = flat ? ceil_div(bn + l.wo - 1, l.wo) : bn / 32;
        const int64_t borders = flat ? ceil_div(rows - 1, l.ho) : 0, wrap = std::max(0, p->hv - l.ho * l.stride_h);
        cells = ((rows - 1) * l.stride_h + borders * wrap + (l.kh - 1) * l.dil_h + 1) * p->wv;
    }
    const bool vec3 = l.kh == 3 && l.kw == 3 && l.dil_w == 1 && *av;
    if (!(point || vec3)) *av = false;
    if (!*av) *bv = false;
    *kind = vec3 ? 9 : point ? 1 : 0;                            // the kernel's TAPS
    int cc = 0;
    if (point) {
        cc = win_point_channels(t.fm * t.fn);
    } else {
        for (int c = 8; c >= (vec3 ? 4 : 2) && !cc; c /= 2)
            if (c * cells <= 2048 && (!vec3 || (c / 2) % t.wk == 0) && (vec3 || int64_t(bm) * c * taps <= 16 * WIN_THREADS)) cc = c;
    }
    if (cc == 0) return false;
    p->cc = cc;
    const size_t partial = size_t(t.wk - 1) * t.wm * t.wn * t.fm * t.fn * 16 * 64 * 4;
    *lds_bytes = std::max(size_t(2 * win_buffer_floats(*kind, cc, cc * taps, bm, bn, *bv)) * 4, partial);
    return *lds_bytes <= 160 * 1024;
}

// CC 0: a 1x1 layer's
template <int TAPS, int CC, bool AV, bool BV>
int launch_tile(int tile, const WinParams &p, size_t lds, hipStream_t s) {
    constexpr int C1 = CC ? CC : win_point_channels(1), C2 = CC ? CC : win_point_channels(2);
    switch (tile) {
        case 0:
            if constexpr (TAPS == 9 && CC == 4) break;
            else return launch_window<1, 1, 4, 1, 1, TAPS, C1, AV, BV>(p, lds, s);
        case 1: return launch_window<1, 4, 1, 1, 1, TAPS, C1, AV, BV>(p, lds, s);
        case 2: return launch_window<2, 2, 1, 1, 1, TAPS, C1, AV, BV>(p, lds, s);
        case 3: return launch_window<2, 2, 1, 1, 2, TAPS, C2, AV, BV>(p, lds, s);
        case 4: return launch_window<2, 2, 1, 2, 2, TAPS, C2, AV, BV>(p, lds, s);
    }
    return fail(TSX_E_INVALID, "conv_f32_window: no tile %d", tile);
}

}  // namespace

int conv_f32_window_tile(const ConvF32Layer &l, double *cycles) {
    const int64_t positions = int64_t(l.n) * l.ho * l.wo;
    // 32-bit byte offsets into every tensor
    const int64_t most = (int64_t(1) << 31) - 64;
    if (int64_t(l.n) * l.c * l.h * l.w * 4 > most || int64_t(l.cout) * l.c * l.kh * l.kw * 4 > most ||
        positions * l.cout * 4 > most)
        return -1;
    if (positions >= (int64_t(1) << 30) || l.pad_top < 0 || l.pad_left < 0) return -1;
    int best = -1;
    double best_cost = 0, best_slow = 1;
    for (int i = 0; i < WIN_TILE_COUNT; ++i)
        for (int flat = 1; flat >= (l.kh * l.kw == 1 ? 1 : 0); --flat) {
            WinParams p{};
            size_t lds = 0;
            int kind = 0;
            bool av, bv;
            if (!plan_tile(l, i, flat != 0, &p, &lds, &kind, &av, &bv)) continue;
            // Time of the busiest CU in fragments of the best tile, by what a fragment costs in each (measured: 3x3 on
            // 28x28 to 112x112 maps, 1x1 on 14x14 and 56x56): K-split tiles pay their reduction, pointwise ones the operand
            // traffic of 32 output channels, and a patch of more than 256 elements per channel halves the chunk.
            static const double per_frag[2][WIN_TILE_COUNT] = {{1.4, 1.0, 1.12, 1.03, 1.08}, {1.45, 1.5, 1.15, 1.0, 1.05}};
            const WinTile &t = WIN_TILES[i];
            const int64_t tiles = int64_t(p.tiles_m) * p.tiles_n, per_cu = ceil_div(tiles, 256);
            const int frags = t.bm() * t.bn() / 1024;
            double cost = double(per_cu) * (frags + 0.2) * per_frag[kind == 1][i];
            if (kind == 9 && p.cc < 8) cost *= 1.12;
            if (kind == 0) cost *= std::max(1.0, double(t.wk) / (p.cc / 2)) * (p.cc < 8 ? 1.12 : 1.0);
            if (best < 0 || cost < best_cost) {
                best = i * 2 + flat;
                best_cost = cost;
                best_slow = kind == 0 && p.cc == 2 && l.kh * l.kw <= 9 ? 1.3 : 1;      // chunks of a few steps
            }
        }
    // the best tile's fragments on four SIMDs: K / 2 MFMAs of 64 cycles each
    if (cycles) *cycles = best_cost * best_slow * l.c * l.kh * l.kw * 8;
    const char *e = std::getenv("TSX_CONV_F32_TILE");
    if (e && e[0]) {
        best = std::atoi(e);
        if (cycles) *cycles = 0;
    }
    return best;
}

void conv_f32_window_tile_size(int tile, int *rows, int *positions) {
    *rows = WIN_TILES[tile / 2].bm();
    *positions = WIN_TILES[tile / 2].bn();
}

int conv_f32_window(const ConvF32Layer &l, int tile, const float *bias, int act, float slope, float padding_value, float *out, hipStream_t stream) {
    WinParams p{};
    size_t lds = 0;
    int kind = 0;
    bool av = false, bv = false;
    if (tile < 0 || tile / 2 >= WIN_TILE_COUNT || !plan_tile(l, tile / 2, tile % 2 != 0, &p, &lds, &kind, &av, &bv))
        return fail(TSX_E_INVALID, "conv_f32_window: tile %d does not suit this layer", tile);
    p.x = l.x_dev;
    p.w = l.w_dev;
    p.bias = bias;
    p.out = out;
    p.padding_value = padding_value;
    p.act = act;
    p.slope = slope;
    p.act_body = int64_t(p.N) * p.M / 4 * 4;
    if (kind == 9)
        return p.cc == 8 ? launch_tile<9, 8, true, false>(tile / 2, p, lds, stream) : launch_tile<9, 4, true, false>(tile / 2, p, lds, stream);
    if (kind == 1)
        return bv ? launch_tile<1, 0, true, true>(tile / 2, p, lds, stream)
               : av ? launch_tile<1, 0, true, false>(tile / 2, p, lds, stream) : launch_tile<1, 0, false, false>(tile / 2, p, lds, stream);
    return p.cc == 8 ? launch_tile<0, 8, false, false>(tile / 2, p, lds, stream)
         : p.cc == 4 ? launch_tile<0, 4, false, false>(tile / 2, p, lds, stream) : launch_tile<0, 2, false, false>(tile / 2, p, lds, stream);
}

}  // namespace tsx
