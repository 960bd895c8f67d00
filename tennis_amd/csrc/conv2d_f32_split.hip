// fp32 convolution on the bf16 matrix cores, for layers of more than some ten million products whose fp32 MFMAs are
// what bounds them (cpu::Conv2DCore, src/kernels/cpu/conv2d_core.cpp:17-119).
//
// v_mfma_f32_32x32x2_f32 gives 64 operations per cycle and SIMD, v_mfma_f32_32x32x16_bf16 1024.  A float of 24
// significant bits is the sum of three bf16 numbers of 8, exactly: x = h + m + l, h the upper half of its bits, m the
// remainder rounded, l what is left of that (m <= 2^-7, l <= 2^-16 of the power of two at or below x).  Of the nine
// products of two such sums eight are formed,
//     x w = h h' + (h m' + m h') + (m m' + h l' + l h') + (m l' + l m'),
// the ninth is below 2^-32 of the product (without m l' and l m', 2^-22, an output that is one product is rounded worse
// than the fp32 MFMA rounds it); each product of two bf16 is exact in the MFMA's fp32 accumulator.  h h' goes to an
// accumulator of its own, the seven small products to a second one, added once at the end: a sum of K terms takes K / 16
// roundings where the fp32 MFMA takes K, and the small terms are not lost beside the large ones.  Measured
// against 64 bits (2-norm; normally distributed and positive operands): 3.9e-8 and 4.0e-8 at K = 32, 6.5e-8 and 5.5e-8 at
// 256, 1.0e-7 and 6.9e-8 at 2304, where the fp32 MFMA kernels have 1.0e-7 and 8.6e-8, 2.9e-7 and 2.5e-7, 4.2e-7 and
// 1.8e-7; on 64 layers that come here by the planner's choice, K from 99 to 7475, 1.2 to 9.2 times less than theirs.
//
// Both operands are split times 2^39, and the result is scaled back: l is a multiple of 2^-23 of x, bf16 ends at 2^-133, and
// times 2^39 the smallest denormal is 2^-110.  So the parts are exact for every number below 2^89, and no part of a product
// that counts is lost.  A tile that meets larger numbers, infinities or NaN, or a sum of 2^50 on its way, is computed again by
// the fp32 MFMA (exact() below): all of them leave an infinity or NaN in the sums they go into.
#include "conv2d_f32_split.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>

namespace tsx {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

struct Parts {
    v4u h, m, l;
};

constexpr float UP = 0x1p39f, DOWN = 0x1p-78f;        // of an operand, of a product

// The three parts of eight floats, times UP, element by element in the order of the MFMA operand; m is NaN where that is
// infinite or NaN.
__device__ __forceinline__ Parts split8(const float (&number)[8]) {
    Parts p;
    float x[8];
    static_for<0, 8>([&](auto jc) { x[decltype(jc)::value] = __fmul_rn(number[decltype(jc)::value], UP); });
    static_for<0, 4>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const unsigned a = __float_as_uint(x[2 * j]), b = __float_as_uint(x[2 * j + 1]);
        p.h[j] = __builtin_amdgcn_perm(b, a, 0x07060302u);
        const float ra = __fsub_rn(x[2 * j], __uint_as_float(a & 0xffff0000u)), rb = __fsub_rn(x[2 * j + 1], __uint_as_float(b & 0xffff0000u));
        const unsigned m = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{ra, rb}), v2b));
        const float qa = __fsub_rn(ra, __uint_as_float(m << 16)), qb = __fsub_rn(rb, __uint_as_float(m & 0xffff0000u));
        p.m[j] = m;
        p.l[j] = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{qa, qb}), v2b));
    });
    return p;
}

// ---- weights [M][C][taps] to MFMA operands [16 channels][tap][32 rows][part][lane][8], zeros behind M and C.
// A workgroup takes 16 channels of 32 rows, through LDS: read as they lie (a lane reading its own 8 channels x taps touches a
// cache line per lane and load: 7.2 us for 256 x 256 x 3 x 3), written a KiB per store instruction.
// No thread splits more than two pieces: few layers have the workgroups to fill the chip, and with 256 threads a 5x5 layer's
// fifty loads and seven pieces of a thread were a chain of 8 us (183 channels to 77; now 5.6), a 3x3 layer's of 5.4 (now 4.2).
constexpr int split_weights_threads(int taps) { return taps == 25 ? 800 : taps == 9 ? 576 : 64; }
template <int TAPS>
__global__ __launch_bounds__(split_weights_threads(TAPS)) void split_weights_kernel(const float *w, int M, int C, int mfrags, v4u *out) {
    constexpr int THREADS = split_weights_threads(TAPS), RUN = 16 * TAPS, PITCH = RUN + 1, LOADS = 32 * RUN / THREADS;
    static_assert(LOADS * THREADS == 32 * RUN && 64 * TAPS % THREADS == 0, "whole rounds");
    __shared__ float rows[32 * PITCH];
    const int tid = threadIdx.x, c0 = blockIdx.y * 16, live = min(16, C - c0) * TAPS;
    float x[LOADS];
    static_for<0, LOADS>([&](auto ic) {
        const int e = tid + THREADS * decltype(ic)::value, k = e % RUN, row = blockIdx.x * 32 + e / RUN;
        x[decltype(ic)::value] = row < M && k < live ? w[(int64_t(row) * C + c0) * TAPS + k] : 0.f;
    });
    static_for<0, LOADS>([&](auto ic) {
        const int e = tid + THREADS * decltype(ic)::value;
        rows[e / RUN * PITCH + e % RUN] = x[decltype(ic)::value];
    });
    __syncthreads();
    v4u *to = out + (int64_t(blockIdx.y) * TAPS * mfrags + blockIdx.x) * 192;
    for (int e = tid; e < 64 * TAPS; e += THREADS) {
        const int lane = e % 64, tap = e / 64;
        float v[8];
        static_for<0, 8>([&](auto jc) { v[decltype(jc)::value] = rows[lane % 32 * PITCH + (8 * (lane / 32) + decltype(jc)::value) * TAPS + tap]; });
        const Parts p = split8(v);
        v4u *dst = to + int64_t(tap) * mfrags * 192 + lane;
        dst[0] = p.h;
        dst[64] = p.m;
        dst[128] = p.l;
    }
}

// A divisor of 1 to 2^30 for numbers below 2^31: with l = ceil(log2 d) and m = ceil(2^(31 + l) / d), which fits in 32 bits,
// n m >> (31 + l) is n / d, since m d < 2^(31 + l) + 2^l.  (The two dozen divisions of a tile's start and end by unknown
// divisors were 2 of its 9 us beside the steps.)
struct Divisor {
    unsigned m, l;
};
Divisor divisor(int64_t d) {
    unsigned l = 0;
    while ((int64_t(1) << l) < d) ++l;
    return {unsigned(((uint64_t(1) << (31 + l)) + uint64_t(d) - 1) / uint64_t(d)), l};
}
__device__ __forceinline__ int quotient(int n, Divisor d) { return int(__umulhi(unsigned(n) << 1, d.m) >> d.l); }

struct SplitParams {
    const float *x, *w32, *bias;
    const void *w;                 // split weights
    float *out;
    int M, N;                      // output channels, positions (n ho wo)
    int n, C, H, W, dil_h, sh, sw, pad_top, pad_left;
    int ho, wo, howo;
    int hv, wv;                    // rows of one image with the padding its windows reach; patch columns
    Divisor by_tiles, by_tiles_m, by_col_tiles, by_seg_rows, by_wo, by_ho, by_howo, by_hv, by_wv;
    int seg, col_tiles;            // a fragment is 32 columns of one row; column tiles per row
    int chunks, mfrags, tiles_m, tiles_n;
    int slices, slice_chunks;      // chunks of one slice; the sums of slice i go to out + i M N
    unsigned w_bytes;
    float padding_value;
    int act;
    float slope;
    int64_t act_body;
};

// A barrier for what has been exchanged through LDS: loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A workgroup of WM x WN wavefronts (8, or two workgroups of 4 per CU) owns 32 WM output channels x 64 WN positions; a
// wavefront's 32 x 64 take 16 MFMAs (512 cycles) per 16 channels and tap for 3 KiB of weights, from L2 straight into
// registers AHEAD steps early, and 6 KiB of activations from LDS.  As in the fp32 form (conv2d_f32_window.hip) a chunk of CC
// channels of the input patch -- the rows and columns the tile's positions read through all taps, padding included -- goes
// to LDS once per element, here in three parts, [part][8 channels][PITCH cells][8], and every tap is a shifted read; a
// thread converts eight channels of a cell at a time while the other wavefront of its SIMD multiplies.  TAPS: 9 (3x3), 25
// (5x5), 1 (the patch is the tile's positions themselves, at any stride).
// Layers of few tiles leave most CUs idle while each tile walks all channels: their chunks go to `slices` of workgroups, whose
// sums another kernel adds in order (2 images of 38x12, 233 channels to 98, 3x3 of stride 2: 47 -> 20 us, of which the fp32
// MFMA kernel's chain of 30 chunks was 1.4 us each; 3 of 30x30, 398 to 31, 5x5: 175 -> 39).  The patches of 768 cells, with one
// workgroup a CU, are strided layers' (6 images of 33x33, 446 to 213, 5x5 of stride 2: 551 us without a tile here, 84).
// What bounds it: the MFMAs at the clock the bf16 matrix cores leave, with conversions, operand reads and weights beside them
// (six products instead of eight, a quarter of the MFMAs less: 55 us instead of 64 on 8 images of 28x28x256 with 256 3x3
// filters).  Against the fp32 MFMAs (us, weights' split included): that layer 84 -> 64, 128 channels at 56x56 77 -> 55, 256 to
// 256 channels 1x1 at 56x56, 32 images, 132 -> 105, 100 to 150 channels 5x5 at 33x41, 4 images, 128 -> 67.
template <int WM, int WN, int TAPS, int PITCH, int CC>
__global__ __launch_bounds__(64 * WM * WN, WM * WN == 4 && PITCH > 384 ? 1 : 2) void conv_f32_split_kernel(SplitParams p) {
    constexpr int THREADS = 64 * WM * WN;
    constexpr int BM = 32 * WM, BN = 64 * WN, KW = TAPS == 9 ? 3 : TAPS == 25 ? 5 : 1;
    constexpr int SUBS = CC / 16, STEPS = SUBS * TAPS;
    constexpr int AHEAD = STEPS <= 4 ? STEPS : 3;
    constexpr int PART = CC / 8 * PITCH * 16, BUFFER = 3 * PART;           // bytes
    constexpr int SLOTS = CC / 8 * PITCH / THREADS;
    static_assert(SUBS >= 1 && CC % 16 == 0 && CC / 8 * PITCH % THREADS == 0 && (TAPS != 1 || PITCH == BN) &&
                      2 * PART + ((SUBS - 1) * 2 * PITCH + KW) * 16 < 65536 && SLOTS <= STEPS,
                  "whole slots, one a step; every operand read within an instruction's offset");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int hf = lane / 32;
    const int wn = wave % WN, wm = wave / WN;

    // Tiles of a slice that share their positions are consecutive, and each XCD takes a contiguous run of tiles: a patch, and
    // where there are many slices their weights, are fetched into one L2.
    const int tiles = p.tiles_m * p.tiles_n, total = tiles * p.slices, per_xcd = (total + 7) / 8;
    const int index = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
    if (int(blockIdx.x >> 3) >= per_xcd || index >= total) return;
    const int slice = quotient(index, p.by_tiles), t = index - slice * tiles;
    const int tn = quotient(t, p.by_tiles_m), m0 = (t - tn * p.tiles_m) * BM;
    const int first_chunk = slice * p.slice_chunks, end_chunk = min(p.chunks, first_chunk + p.slice_chunks);

    // ---- positions: flat over the batch, or segments (image, first row inside it, first column)
    const int seg_rows = (p.ho + BN / 32 - 1) / (BN / 32), seg_tile = p.seg ? quotient(tn, p.by_col_tiles) : 0, seg_img = quotient(seg_tile, p.by_seg_rows);
    const int seg_row = (seg_tile - seg_img * seg_rows) * (BN / 32);
    const int col0 = p.seg ? (tn - seg_tile * p.col_tiles) * 32 : 0;
    auto decode = [&](int q, int &row, int &col) -> bool {                 // tile position -> batch-wide output row, column
        if (p.seg) {
            row = seg_img * p.ho + seg_row + q / 32;
            col = col0 + q % 32;
            return seg_row + q / 32 < p.ho && col < p.wo;
        }
        const int pos = tn * BN + q;
        row = quotient(pos, p.by_wo);
        col = pos - row * p.wo;
        return pos < p.N;
    };
    auto virtual_row = [&](int row) { const int img = quotient(row, p.by_ho); return img * p.hv + (row - img * p.ho) * p.sh; };
    const int vr0 = virtual_row(p.seg ? seg_img * p.ho + seg_row : quotient(tn * BN, p.by_wo));

    // ---- patch bookkeeping: slot i of a thread is cell (tid + 512 i) % PITCH of the chunk's eight channels (tid + 512 i) / PITCH
    constexpr unsigned NOWHERE = 0x80000000u;                              // beyond any buffer: loads 0, stores nothing
    const unsigned plane = unsigned(p.H) * unsigned(p.W);
    unsigned x_off[SLOTS];                                                 // NOWHERE: the cell is padding
    static_for<0, SLOTS>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int e = tid + THREADS * i, octet = e / PITCH, cell = e % PITCH;
        int img, h, w;
        bool in = true;
        if (TAPS == 1) {
            const int pos = tn * BN + cell;
            img = quotient(pos, p.by_howo);
            const int r = pos - img * p.howo, oh = quotient(r, p.by_wo);
            in = pos < p.N;
            h = oh * p.sh - p.pad_top;
            w = (r - oh * p.wo) * p.sw - p.pad_left;
        } else {
            const int pr = quotient(cell, p.by_wv), v = vr0 + pr;
            img = quotient(v, p.by_hv);
            in = img < p.n;                                                // cells behind the tile's patch: loaded, never used
            h = v - img * p.hv - p.pad_top;
            w = cell - pr * p.wv + col0 * p.sw - p.pad_left;
        }
        in = in && h >= 0 && h < p.H && w >= 0 && w < p.W;
        x_off[i] = in ? ((unsigned(img) * unsigned(p.C) + unsigned(8 * octet)) * plane + unsigned(h * p.W + w)) * 4u : NOWHERE;
    });

    auto x_octet = [&](int i) {                // computed where it is used, not kept over the whole loop
        int e = tid + THREADS * i;
        asm volatile("" : "+v"(e));
        return e / PITCH;
    };
    float x_reg[SLOTS][8];
    const int x_bytes = int(int64_t(p.n) * p.C * plane * 4);               // below 2 GiB
    // Two forms of what follows, neither with a branch between the MFMAs.  0: eight channels are there or not, padding is 0.
    // 1: any channels and padding value.
    const bool ragged = p.C % 8 != 0 || p.padding_value != 0.f;
    // Channels FROM to TO of the chunk for slot i.  A chunk behind the last one has no channel, and reads nothing:
    // its offsets are beyond the buffer (whose size stays above every channel's scalar offset, from which the hardware counts).
    auto load_patch = [&](auto form, auto ic, auto from, auto to, int chunk) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        const bool live = chunk < end_chunk;
        const int c0 = live ? chunk * CC : 0, at = c0 * int(plane) * 4;
        const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(p.x) + at), 0, x_bytes - at, 0x00020000);
        const int left = (live ? p.C - c0 : 0) - 8 * x_octet(i);
        unsigned base = x_off[i];
        if constexpr (decltype(form)::value != 0) asm volatile("" : "+v"(base));      // no sums of it kept either
        static_for<decltype(from)::value, decltype(to)::value>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            if constexpr (decltype(form)::value == 0) {
                x_reg[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, left > 0 ? int(base) : int(NOWHERE), j * int(plane) * 4, 0));
            } else {                           // (the sum of an offset beyond the buffer and a channel's stays beyond it)
                const unsigned off = base + unsigned(j) * plane * 4u;
                x_reg[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, int(j < left ? off : NOWHERE), 0, 0));
            }
        });
    };
    auto store_patch = [&](auto form, auto ic, int chunk, int at) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (decltype(form)::value != 0) {
            const int channels = p.C - chunk * CC - 8 * x_octet(i), left = x_off[i] == NOWHERE ? channels : 0;
            static_for<0, 8>([&](auto jc) { x_reg[i][decltype(jc)::value] = decltype(jc)::value < left ? p.padding_value : x_reg[i][decltype(jc)::value]; });
        }
        const Parts s = split8(x_reg[i]);
        char *to = lds + at + (tid + THREADS * i) * 16;
        *reinterpret_cast<v4u *>(to) = s.h;
        *reinterpret_cast<v4u *>(to + PART) = s.m;
        *reinterpret_cast<v4u *>(to + 2 * PART) = s.l;
    };

    // ---- operands.  Step (sub, tap) of a chunk takes channels 16 sub ... of it.
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.w), 0, int(p.w_bytes), 0x00020000);
    const int w_off = min(m0 / 32 + wm, p.mfrags - 1) * 3072 + lane * 16, w_step = p.mfrags * 3072;
    struct A { v4u part[3]; } a[AHEAD];
    struct B { v4u part[2][3]; } b;
    auto load_weights = [&](auto sc, int chunk) __attribute__((always_inline)) {      // step sc of the chunk, its steps beyond STEPS in the next
        constexpr int s = decltype(sc)::value % STEPS, over = decltype(sc)::value / STEPS, sub = s / TAPS, tap = s % TAPS;
        const int q = ((min(chunk + over, end_chunk - 1) * (CC / 16) + sub) * TAPS + tap) * w_step;
        static_for<0, 3>([&](auto pc) {
            constexpr int part = decltype(pc)::value;
            a[s % AHEAD].part[part] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + part * 1024, q, 0));
        });
    };
    int b_at[2];                               // LDS address of this lane's positions in the patch
    const int row_bytes = p.dil_h * p.wv * 16; // from one kernel row to the next
    static_for<0, 2>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const int q = (wn * 2 + j) * 32 + lane % 32;
        int row, col;
        const bool ok = decode(q, row, col);
        const int cell = TAPS == 1 ? q : ok ? (virtual_row(row) - vr0) * p.wv + (col - col0) * p.sw : 0;
        b_at[j] = (hf * PITCH + cell) * 16;
    });
    auto read = [&](auto sc, int at) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value, sub = s / TAPS, tap = s % TAPS;
        B v;
        static_for<0, 6>([&](auto ec) {
            constexpr int j = decltype(ec)::value / 3, part = decltype(ec)::value % 3;
            v.part[j][part] = *reinterpret_cast<const v4u *>(lds + (b_at[j] + (at + tap / KW * row_bytes)) + part * PART + (2 * sub * PITCH + tap % KW) * 16);
        });
        return v;
    };
    v16f sum[2], large[2], small[2];
    auto multiply = [&](const A &w, const B &v) __attribute__((always_inline)) {
        const auto mfma = [&](auto wc, auto vc, v16f(&to)[2]) __attribute__((always_inline)) {
            static_for<0, 2>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                to[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, w.part[decltype(wc)::value]),
                                                                __builtin_bit_cast(v8b, v.part[j][decltype(vc)::value]), to[j], 0, 0, 0);
            });
        };
        const std::integral_constant<int, 0> h;
        const std::integral_constant<int, 1> m;
        const std::integral_constant<int, 2> l;
        mfma(m, l, small);
        mfma(l, m, small);
        mfma(l, h, small);
        mfma(h, l, small);
        mfma(m, m, small);
        mfma(m, h, small);
        mfma(h, m, small);
        mfma(h, h, large);
    };

    // The steps of a chunk: the next step's activations are read under a step's MFMAs, the weights AHEAD steps early.  The next
    // chunk's patch is stored slot by slot, spread over the steps, and the one behind it requested into the registers that
    // become free, a few loads a step (all at once they would hold up the weights behind them).  The barrier in front of the
    // last step: the other buffer is stored, and this one's last reads have returned.
    auto run = [&](auto form) __attribute__((always_inline)) {
        const std::integral_constant<int, 0> none;
        const std::integral_constant<int, 8> all;
        static_for<0, SLOTS>([&](auto ic) { load_patch(form, ic, none, all, first_chunk); });
        static_for<0, AHEAD>([&](auto sc) { load_weights(sc, first_chunk); });
        static_for<0, SLOTS>([&](auto ic) { store_patch(form, ic, first_chunk, 0); });
        static_for<0, SLOTS>([&](auto ic) { load_patch(form, ic, none, all, first_chunk + 1); });
        sum[0] = sum[1] = small[0] = small[1] = v16f{};
        lds_barrier();
        b = read(none, 0);
        int chunk = first_chunk, now = 0;
        do {
            const int next = BUFFER - now;
            large[0] = large[1] = v16f{};
            static_for<0, STEPS>([&](auto sc) {
                constexpr int s = decltype(sc)::value, slot = s * SLOTS / STEPS, first = (slot * STEPS + SLOTS - 1) / SLOTS;
                constexpr int steps = ((slot + 1) * STEPS + SLOTS - 1) / SLOTS - first;      // from this slot's store to the next one's
                const std::integral_constant<int, slot> ic;
                if constexpr (s + 1 == STEPS) {
                    if constexpr (s == first) store_patch(form, ic, chunk + 1, next);
                    lds_barrier();
                }
                B after;
                if constexpr (s + 1 < STEPS) after = read(std::integral_constant<int, s + 1>{}, now);
                else after = read(none, next);
                multiply(a[s % AHEAD], b);
                load_weights(std::integral_constant<int, s + AHEAD < STEPS ? s + AHEAD : STEPS + s % AHEAD>{}, chunk);
                if constexpr (s == first && s + 1 < STEPS) store_patch(form, ic, chunk + 1, next);
                load_patch(form, ic, std::integral_constant<int, (s - first) * 8 / steps>{}, std::integral_constant<int, (s - first + 1) * 8 / steps>{}, chunk + 2);
                b = after;
                // vector instructions go between the MFMAs, which take 32 cycles each
                static_for<0, 16>([&](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, s == first ? 6 : 3, 0);
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                });
                __builtin_amdgcn_sched_barrier(0);
            });
            sum[0] += large[0];
            sum[1] += large[1];
            now = next;
        } while (++chunk < end_chunk);
    };
    if (ragged) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 0>{});
    sum[0] += small[0];
    sum[1] += small[1];
    int late = __lane_id();
    asm volatile("" : "+v"(late));             // nothing of what follows is kept over the loop: positions are decoded again
    const int in_row = late % 32, half = late / 32;

    // The tile on the fp32 MFMA, operands straight from the tensors: products in the order of the weights (channel, tap), one
    // rounding each, every second one in the wavefront's upper half.
    auto exact = [&]() __attribute__((always_inline)) {
        constexpr int BLOCK = 8;               // MFMAs per fragment whose operands are requested together
        const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x), 0, x_bytes, 0x00020000);
        const auto wr32 = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.w32), 0, p.M * p.C * TAPS * 4, 0x00020000);
        const int w_row = min(m0 + wm * 32 + in_row, p.M - 1) * p.C * TAPS, products = min(p.C, end_chunk * CC) * TAPS;
        unsigned first[2], inside[2];          // element of the first tap in the first channel; a bit per tap
        static_for<0, 2>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            int row, col;
            const bool ok = decode((wn * 2 + j) * 32 + in_row, row, col);
            const int img = quotient(row, p.by_ho), h = (row - img * p.ho) * p.sh - p.pad_top, w = col * p.sw - p.pad_left;
            first[j] = unsigned(img) * unsigned(p.C) * plane + unsigned(h * p.W + w);
            inside[j] = 0;
            for (int tap = 0; tap < TAPS; ++tap) {
                const int y = h + tap / KW * p.dil_h, x = w + tap % KW;
                inside[j] |= unsigned(ok && y >= 0 && y < p.H && x >= 0 && x < p.W) << tap;
            }
        });
        sum[0] = sum[1] = v16f{};
        for (int k0 = first_chunk * CC * TAPS; k0 < products; k0 += 2 * BLOCK) {
            float w[BLOCK], x[2][BLOCK];
            unsigned at[2][BLOCK];
            static_for<0, BLOCK>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                const int k = k0 + 2 * e + half, ch = k / TAPS, tap = k % TAPS;
                const bool there = k < products;
                w[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wr32, there ? (w_row + k) * 4 : int(NOWHERE), 0, 0));
                static_for<0, 2>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const unsigned off = (first[j] + unsigned(ch) * plane + unsigned(tap / KW * p.dil_h * p.W + tap % KW)) * 4u;
                    at[j][e] = !there ? NOWHERE + 4 : inside[j] >> tap & 1u ? off : NOWHERE;
                    x[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, int(at[j][e]), 0, 0));
                });
                __builtin_amdgcn_sched_barrier(0);      // a few conditions at a time: scalar registers
            });
            static_for<0, 2 * BLOCK>([&](auto ec) {
                constexpr int e = decltype(ec)::value / 2, j = decltype(ec)::value % 2;
                sum[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[e], at[j][e] == NOWHERE ? p.padding_value : x[j][e], sum[j], 0, 0, 0);
            });
        }
    };
    bool odd = false;
    static_for<0, 32>([&](auto rc) {
        const float v = sum[decltype(rc)::value / 16][decltype(rc)::value % 16];
        odd |= !(__builtin_fabsf(v) < __builtin_inff());
        sum[decltype(rc)::value / 16][decltype(rc)::value % 16] = __fmul_rn(v, DOWN);
    });
    // (behind the last step's barrier no one uses what is read from LDS; __syncthreads_or would keep a register over the loop)
    int *const odd_wave = reinterpret_cast<int *>(lds);
    const int any = __any(odd);
    if (late == 0) odd_wave[wave] = any;
    lds_barrier();
    int odd_tile = 0;
    static_for<0, THREADS / 64>([&](auto wc) { odd_tile |= odd_wave[decltype(wc)::value]; });
    if (__builtin_amdgcn_readfirstlane(odd_tile)) exact();

    // ---- bias values of the tile's rows, requested together
    float bias[16];
    static_for<0, 16>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        bias[r] = p.bias ? p.bias[min(m0 + wm * 32 + 8 * (r / 4) + 4 * half + r % 4, p.M - 1)] : 0.f;
    });
    // A lane's element of a row is its own offset plus a uniform one; 32-bit offsets, the output is below 2 GiB.
    const auto out = __builtin_amdgcn_make_buffer_rsrc(p.out + int64_t(slice) * p.M * p.N, 0, int(int64_t(p.M) * p.N * 4), 0x00020000);
    const bool body = p.act_body == int64_t(p.M) * p.N;      // no element behind the activation's SIMD body
    static_for<0, 2>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        int row, col;
        const bool ok = decode((wn * 2 + j) * 32 + in_row, row, col);
        const int img = quotient(row, p.by_ho);
        const int base = img * p.M * p.howo + (row - img * p.ho) * p.wo + col + (m0 + wm * 32 + 4 * half) * p.howo;
        static_for<0, 16>([&](auto rc) {
            constexpr int r = decltype(rc)::value, up = 8 * (r / 4) + r % 4;
            float v = sum[j][r];
            if (p.bias) v = __fadd_rn(v, bias[r]);
            v = apply_act_basic(v, p.act, p.slope, body || base + up * p.howo < p.act_body);
            const bool in = ok && m0 + wm * 32 + 4 * half + up < p.M;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), out, in ? base * 4 : int(NOWHERE), up * p.howo * 4, 0);
        });
    });
}

// ---- slices' sums [slice][output] to the output, in the order of the slices.  VEC: 4 outputs at a time, which start a channel
// or lie inside one.
struct SliceParams {
    const float *sums, *bias;
    float *out;
    unsigned total, howo, M;
    int slices, act;
    float slope;
    int64_t act_body;
};

template <int VEC>
__global__ __launch_bounds__(256) void sum_slices_kernel(SliceParams p) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const unsigned at = (blockIdx.x * 256 + threadIdx.x) * VEC;
    if (at >= p.total) return;
    const float bias = p.bias ? p.bias[at / p.howo % p.M] : 0.f;
    auto slice = [&](int s) __attribute__((always_inline)) { return *reinterpret_cast<const vec *>(p.sums + int64_t(s) * p.total + at); };
    vec sum = slice(0);
    int s = 1;
    for (; s + 4 <= p.slices; s += 4) {        // four requests in flight
        vec q[4];
        static_for<0, 4>([&](auto ic) { q[decltype(ic)::value] = slice(s + decltype(ic)::value); });
        static_for<0, 4>([&](auto ic) { sum += q[decltype(ic)::value]; });
    }
    for (; s < p.slices; ++s) sum += slice(s);
    static_for<0, VEC>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const float v = p.bias ? __fadd_rn(sum[i], bias) : sum[i];
        sum[i] = apply_act_basic(v, p.act, p.slope, int64_t(at) + i < p.act_body);
    });
    *reinterpret_cast<vec *>(p.out + at) = sum;
}

// ---- tiles.  Each with the patch pitches it is built for, smallest first.
struct SplitTile {
    int wm, wn, taps, pitch, cc;
    int (*launch)(const SplitParams &, hipStream_t);
    int bm() const { return 32 * wm; }
    int bn() const { return 64 * wn; }
};

template <int WM, int WN, int TAPS, int PITCH, int CC>
int launch_split(const SplitParams &p, hipStream_t stream) {
    auto kernel = conv_f32_split_kernel<WM, WN, TAPS, PITCH, CC>;
    constexpr size_t lds_bytes = 2 * 3 * CC / 8 * PITCH * 16;
    static_assert(lds_bytes <= 159 * 1024, "LDS of a compute unit");
    if (lds_bytes > 65536) {                   // dynamic LDS beyond 64 KiB is granted per kernel and device
        static std::atomic<bool> granted[64];
        int dev = 0;
        TSX_HIP(hipGetDevice(&dev));
        if (dev >= 64 || !granted[dev].load()) {
            TSX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_bytes)));
            if (dev < 64) granted[dev].store(true);
        }
    }
    const int total = p.tiles_m * p.tiles_n * p.slices;
    hipLaunchKernelGGL(kernel, dim3(unsigned((total + 7) / 8 * 8)), dim3(64 * WM * WN), lds_bytes, stream, p);
    TSX_LAUNCH_CHECK("conv_f32_split_kernel");
    return 0;
}

template <int WM, int WN, int TAPS, int PITCH, int CC>
constexpr SplitTile split_tile() { return {WM, WN, TAPS, PITCH, CC, launch_split<WM, WN, TAPS, PITCH, CC>}; }

const SplitTile SPLIT_TILES[] = {
    split_tile<2, 2, 9, 256, 16>(), split_tile<2, 2, 9, 384, 16>(), split_tile<4, 1, 9, 256, 16>(), split_tile<4, 1, 9, 384, 16>(), split_tile<4, 2, 9, 512, 16>(),
    split_tile<2, 2, 25, 384, 16>(), split_tile<4, 1, 25, 256, 16>(), split_tile<4, 1, 25, 384, 16>(),
    split_tile<4, 1, 1, 64, 64>(), split_tile<2, 2, 1, 128, 32>(),
    split_tile<4, 2, 9, 768, 16>(), split_tile<2, 2, 9, 768, 16>(), split_tile<4, 1, 9, 768, 16>(),
    split_tile<4, 2, 25, 768, 16>(), split_tile<2, 2, 25, 768, 16>(), split_tile<4, 1, 25, 768, 16>(),
};
constexpr int SPLIT_TILE_COUNT = int(sizeof(SPLIT_TILES) / sizeof(SPLIT_TILES[0]));

// The launch of one layer with one tile; false if the tile is not the layer's or its patch does not fit.
bool plan_tile(const ConvF32Layer &l, int tile, bool flat, SplitParams *p) {
    const SplitTile &t = SPLIT_TILES[tile];
    const int bn = t.bn(), k = t.taps == 9 ? 3 : t.taps == 25 ? 5 : 1;
    if (l.kh != k || l.kw != k || l.dil_w != 1 || (k == 1 && !flat)) return false;
    p->M = l.cout;
    p->N = int(int64_t(l.n) * l.ho * l.wo);
    p->n = l.n; p->C = l.c; p->H = l.h; p->W = l.w;
    p->dil_h = l.dil_h; p->sh = l.stride_h; p->sw = l.stride_w;
    p->pad_top = l.pad_top; p->pad_left = l.pad_left;
    p->ho = l.ho; p->wo = l.wo; p->howo = l.ho * l.wo;
    p->hv = (l.ho - 1) * l.stride_h + (k - 1) * l.dil_h + 1;
    p->chunks = int(ceil_div(l.c, t.cc));
    p->mfrags = int(ceil_div(l.cout, 32));
    p->tiles_m = int(ceil_div(l.cout, t.bm()));
    p->seg = !flat;
    p->col_tiles = flat ? 1 : int(ceil_div(l.wo, 32));
    p->wv = (flat ? l.wo - 1 : 31) * l.stride_w + k;
    const int64_t tiles_n = flat ? ceil_div(p->N, bn) : int64_t(l.n) * ceil_div(l.ho, bn / 32) * p->col_tiles;
    if (tiles_n * p->tiles_m >= (int64_t(1) << 22)) return false;
    p->tiles_n = int(tiles_n);
    if (k > 1) {
        // rows of the largest patch: output rows a tile touches, and per image border it crosses the padding rows between
        const int64_t rows = flat ? ceil_div(bn + l.wo - 1, l.wo) : bn / 32;
        const int64_t borders = flat ? ceil_div(rows - 1, l.ho) : 0, wrap = std::max(0, p->hv - l.ho * l.stride_h);
        if (((rows - 1) * l.stride_h + borders * wrap + (k - 1) * l.dil_h + 1) * p->wv > t.pitch) return false;
    }
    const int64_t w_bytes = int64_t(p->chunks) * (t.cc / 16) * t.taps * p->mfrags * 3072;
    if (w_bytes > (int64_t(1) << 31) - 64) return false;
    p->w_bytes = unsigned(w_bytes);
    return true;
}

// What a launch needs beyond the plan (not a part of it: nine divisions of 64 bits for each of some fifteen tiles were half of its time).
void set_divisors(SplitParams *p, int bn) {
    p->by_tiles = divisor(int64_t(p->tiles_n) * p->tiles_m);
    p->by_tiles_m = divisor(p->tiles_m);
    p->by_col_tiles = divisor(p->col_tiles);
    p->by_seg_rows = divisor(ceil_div(p->ho, bn / 32));
    p->by_wo = divisor(p->wo);
    p->by_ho = divisor(p->ho);
    p->by_howo = divisor(p->howo);
    p->by_hv = divisor(p->hv);
    p->by_wv = divisor(p->wv);
}

}  // namespace

ConvF32Split conv_f32_split_choose(const ConvF32Layer &l, size_t workspace_bytes) {
    ConvF32Split best{-1, 0, 0., 1};
    // "0": never; a number: that tile wherever it suits, in one slice or, "number/slices", in so many where there are the chunks
    // and the workspace (tests)
    const char *e = std::getenv("TSX_CONV_F32_SPLIT");
    if (e && e[0] == '0' && !e[1]) return best;
    const int only = e && e[0] ? std::atoi(e) - 1 : -1;
    const char *slash = only >= 0 ? std::strchr(e, '/') : nullptr;
    const int only_slices = slash ? std::max(1, std::atoi(slash + 1)) : 1;
    const int64_t most = (int64_t(1) << 31) - 64;              // 32-bit byte offsets into every tensor
    const int64_t positions = int64_t(l.n) * l.ho * l.wo;
    if (int64_t(l.n) * l.c * l.h * l.w * 4 > most || positions * l.cout * 4 > most || positions >= (int64_t(1) << 30) || l.pad_top < 0 || l.pad_left < 0)
        return best;
    for (int i = 0; i < SPLIT_TILE_COUNT; ++i)
        for (int flat = 1; flat >= 0; --flat) {
            SplitParams p{};
            if ((only >= 0 && i * 2 + flat != only) || !plan_tile(l, i, flat != 0, &p)) continue;
            if (p.w_bytes > workspace_bytes) continue;
            const SplitTile &t = SPLIT_TILES[i];
            // Time in us: the launches; by the tiles of a CU and their chunks the steps of MFMAs (of eight wavefronts two to a SIMD)
            // and the conversion of the patch, twice as much where channels are no whole eights and each is looked at; the tiles'
            // start and end, of which little is seen where a CU holds two workgroups; the last, partly empty round; the weights
            // and the output.  Slices cost their sums' way through memory and one more launch.  Fitted to 23 000 combinations of tile
            // and slices on 800 layers of 0.01 to 15 GFLOP, which it meets by 5 % (rms); the combinations it picks take 0.5 %
            // longer than the fastest on average, one in a hundred more than 7 %.
            const bool eight = t.wm * t.wn == 8, alone = t.pitch > 384, whole = l.c % 8 == 0;
            const double sums = double(positions) * l.cout * 4e-6, weights = double(l.cout) * l.c * t.taps * 1e-6;
            const int steps = t.cc / 16 * t.taps, all = p.tiles_m * p.tiles_n;
            const double start = alone ? eight ? 3.2 : 4.6 : 1.35, patch = (t.taps == 1 ? t.bn() : t.pitch) * (t.cc / 16) * (whole ? 0.0010 : 0.00215);
            const double tile_cost = t.pitch * 1e-4 + t.wn * 0.1;      // of equal ones the smaller patch, the taller tile
            // every number of slices that leaves none empty, by the chunks of each, as long as what only grows with it stays
            // below the best: twenty tiles of 128 chunks are planned in 3 us
            for (int each = p.chunks; each > 0; --each) {
                const int slices = (p.chunks + each - 1) / each;
                each = (p.chunks + slices - 1) / slices;
                const double tiles = double(all) * slices / 256;
                const double step = (eight ? 0.488 : tiles <= 1 ? 0.29 : 0.27) * (t.taps == 1 ? 0.9 : 1);
                const double rest = 9.2 + 2.6 * weights + 0.18 * sums + (slices > 1 ? 1.8 + 0.4 * slices * sums : 0) + tile_cost;
                const size_t bytes = p.w_bytes + (slices > 1 ? size_t(slices) * size_t(positions) * l.cout * 4 : 0);
                if (bytes > workspace_bytes) break;
                if (only >= 0) {
                    if (slices <= int(ceil_div(p.chunks, ceil_div(p.chunks, only_slices)))) best = {i * 2 + flat, bytes, 0., slices};
                    continue;
                }
                if (best.tile >= 0 && rest + tiles * start + double(all) / 256 * p.chunks * (steps * (eight || tiles > 1 ? step : step / 0.29 * 0.27) + patch) >= best.us) break;
                const double rounds = tiles <= 1 ? 0.8 + 0.2 * tiles : tiles + (alone ? 1 : 0.69) * (int((int64_t(all) * slices + 255) / 256) - tiles);
                const double lone = eight || alone ? 1 + 0.12 * std::clamp((tiles - 1) / 3, 0., 1.) : 1;      // a CU's only workgroup, one after the other
                const double us = rest + rounds * lone * (each * (steps * step + patch) + start);
                if (best.tile < 0 || us < best.us) best = {i * 2 + flat, bytes, us, slices};
            }
        }
    return best;
}

void conv_f32_split_tile_size(int tile, int *rows, int *positions, int *patch) {
    *rows = SPLIT_TILES[tile / 2].bm();
    *positions = SPLIT_TILES[tile / 2].bn();
    *patch = SPLIT_TILES[tile / 2].pitch;
}

int conv_f32_split(const ConvF32Layer &l, const ConvF32Split &choice, const float *bias, int act, float slope, float padding_value, float *out,
                   void *workspace, hipStream_t stream) {
    SplitParams p{};
    const int tile = choice.tile, slices = choice.slices;
    if (tile < 0 || tile / 2 >= SPLIT_TILE_COUNT || !plan_tile(l, tile / 2, tile % 2 != 0, &p))
        return fail(TSX_E_INVALID, "conv_f32_split: tile %d does not suit this layer", tile);
    const SplitTile &t = SPLIT_TILES[tile / 2];
    set_divisors(&p, t.bn());
    const dim3 grid(unsigned(p.mfrags), unsigned(p.chunks * (t.cc / 16)));
    const auto pack = t.taps == 9 ? split_weights_kernel<9> : t.taps == 25 ? split_weights_kernel<25> : split_weights_kernel<1>;
    hipLaunchKernelGGL(pack, grid, dim3(unsigned(split_weights_threads(t.taps))), 0, stream, l.w_dev, l.cout, l.c, p.mfrags, static_cast<v4u *>(workspace));
    TSX_LAUNCH_CHECK("split_weights_kernel");
    p.x = l.x_dev;
    p.w32 = l.w_dev;
    p.w = workspace;
    p.padding_value = padding_value;
    p.slices = slices;
    p.slice_chunks = int(ceil_div(p.chunks, slices));
    const int64_t total = int64_t(p.N) * p.M, act_body = total / 4 * 4;
    if (slices == 1) {
        p.bias = bias;
        p.out = out;
        p.act = act;
        p.slope = slope;
        p.act_body = act_body;
        return t.launch(p, stream);
    }
    p.out = reinterpret_cast<float *>(static_cast<char *>(workspace) + p.w_bytes);
    p.act = TSX_ACT_NONE;
    p.act_body = total;
    const int rc = t.launch(p, stream);
    if (rc) return rc;
    const SliceParams q{p.out, bias, out, unsigned(total), unsigned(p.howo), unsigned(p.M), slices, act, slope, act_body};
    const bool vec = p.howo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    hipLaunchKernelGGL(vec ? sum_slices_kernel<4> : sum_slices_kernel<1>, dim3(unsigned(ceil_div(total, vec ? 1024 : 256))), dim3(256), 0, stream, q);
    TSX_LAUNCH_CHECK("sum_slices_kernel");
    return 0;
}

}  // namespace tsx
