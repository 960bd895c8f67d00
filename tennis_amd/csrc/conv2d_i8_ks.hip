// int8 convolution with K split over the wavefronts of a workgroup: small maps, and 1x1 layers with a stride.
// Same arithmetic, staged input, packed weights and epilogue as conv2d_i8_ws.hip (exact int32 sums of
// cpu::Conv2DQuantizedCore, src/kernels/cpu/quantized/conv2d_quantized_core.cpp:18-147).
//
// The window-stationary kernel gives each wavefront all of K for its output channels; on a 7x7 map that is 72 K-steps in
// a row on eight workgroups, each step an L2 latency's share.  Here the four wavefronts of a workgroup own the same R MT
// channels x R positions and a quarter of the K-steps.  Nothing is shared before the end, so there is no window, no barrier
// and no LDS in front of the MFMAs: weights and activations go from L2 straight into registers (a 1x1 layer's stride, or
// a tap, is an offset), D K-steps of them requested before the first is used, and the epilogue's scales, biases and
// residual values right behind them: a layer is one round trip to memory, the MFMAs, and one exchange through LDS in
// which the four partial sums meet (int32: any order is exact).
#include "conv2d_i8_ks.hpp"

#include <cstdlib>

namespace tsx {
namespace {

struct KsParams : EpiParams {
    const int8_t *xs;      // staged activations [n][hs][ws][cp]
    const int8_t *wp;      // packed weights [ks][coutp/32][2 halves][64 lanes][16]
    int cout, frags, positions, wo, howo, hs, ws, cp;
    int sh, sw, kw, taps, cblocks, ksteps;
    int row_bytes, col_bytes;      // from one tap to the next
    unsigned cblocks_magic, kw_magic, wo_magic, howo_magic, tiles_n_magic;
    int tiles_m, tiles_n;
    int rounds;                    // of D K-steps per wavefront
};

// (udiv, with the divisor 1 that most of these are taken without a division as well)
__device__ __forceinline__ int quotient(int n, int d, unsigned magic) { return d == 1 ? n : udiv(n, d, magic); }

constexpr int W = 4;               // wavefronts of a workgroup

template <int R, int MT, int D, bool MISHX>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2))) void conv_i8_ks_kernel(KsParams p) {
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];   // partial sums [unit][wavefront][lane][4]
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), in = lane % R, part = lane / R;
    // Tiles that read the same weights are consecutive, and each XCD takes a contiguous run of tiles: the weights,
    // most of a small map's bytes, are fetched into one L2.
    const int total = p.tiles_m * p.tiles_n, per_xcd = (total + 7) / 8;
    const int t = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
    if (int(blockIdx.x >> 3) >= per_xcd || t >= total) return;
    const int tm = quotient(t, p.tiles_n, p.tiles_n_magic), m0 = tm * (R * MT), n0 = (t - tm * p.tiles_n) * R;

    // ---- this lane's position, and where its pixel lies from the tile's first image on: 32 bits
    const int img0 = quotient(n0, p.howo, p.howo_magic);
    const int8_t *x_base = p.xs + int64_t(img0) * p.hs * p.ws * p.cp;
    const int pos = n0 + in, at = min(pos, p.positions - 1);               // beyond the last: computed, never stored
    const int img = quotient(at, p.howo, p.howo_magic), rem = at - img * p.howo, oh = quotient(rem, p.wo, p.wo_magic);
    const unsigned b_off = unsigned((((img - img0) * p.hs + oh * p.sh) * p.ws + (rem - oh * p.wo) * p.sw) * p.cp + part * 16);
    // ---- operands.  K-steps in the order (tap, channel block), a run of them per wavefront: two channel blocks of a pixel
    // share a cache line.
    // Lane l supplies row / column l % R and 16 bytes of K, group l / R, of v_mfma_i32_32x32x32_i8 or _16x16x64_i8.
    constexpr int HALVES = R / 16;             // MFMAs (and loads of an operand) per K-step: K of 32 or 64
    const unsigned a_off = R == 32 ? unsigned(lane * 16) : unsigned((part / 2) * 1024 + (part % 2) * 512 + in * 16);
    v4i a[D][MT][HALVES], b[D][HALVES];
    const int k_first = p.ksteps * wave / W, k_end = p.ksteps * (wave + 1) / W;
    auto load = [&](auto slot, int k) __attribute__((always_inline)) {
        constexpr int s = decltype(slot)::value;
        k = min(k, p.ksteps - 1);                                          // beyond the last K-step: its lines again
        const int tap = quotient(k, p.cblocks, p.cblocks_magic), cb = k - tap * p.cblocks, kh = quotient(tap, p.kw, p.kw_magic);
        const int8_t *xk = x_base + (kh * p.row_bytes + (tap - kh * p.kw) * p.col_bytes + cb * 64);
        const int8_t *wk = p.wp + int64_t(cb * p.taps + tap) * p.frags * 2048;
        static_for<0, MT>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int row = min(m0 + i * R, p.frags * 32 - R);             // rows beyond the packed ones: computed, never stored
            const int8_t *wi = wk + row / 32 * 2048 + row % 32 * 16;
            unsigned off = a_off;
            asm volatile("" : "+v"(off));                                  // (scalar base + lane offset: no address arithmetic)
            static_for<0, HALVES>([&](auto hc) { a[s][i][decltype(hc)::value] = *reinterpret_cast<const v4i *>(wi + off + decltype(hc)::value * 1024); });
        });
        unsigned off = b_off;
        asm volatile("" : "+v"(off));
        static_for<0, HALVES>([&](auto hc) { b[s][decltype(hc)::value] = *reinterpret_cast<const v4i *>(xk + off + decltype(hc)::value * 32); });
    };
    static_for<0, D>([&](auto sc) { load(sc, k_first + decltype(sc)::value); });

    // ---- epilogue units: 4 consecutive channels (accumulator registers 4g..4g+3) by 64 / R by a fragment's R positions.  A
    // wavefront takes U of them, all of one fragment; with more wavefronts than units the last ones take none.  What a
    // unit's values meet is requested now.
    constexpr int PER_FRAG = R == 32 ? 4 : 1, UNITS = PER_FRAG * MT, U = UNITS >= W ? UNITS / W : 1;
    static_assert((UNITS % W == 0 || W % UNITS == 0) && U <= PER_FRAG, "whole units per wavefront, of one fragment");
    const bool mine = wave * U < UNITS;
    const bool want_q = p.out_i8 || p.st_out, values = p.out_f32 || want_q;
    const int frag = wave * U / PER_FRAG;
    const int co_first = m0 + frag * R + wave * U % PER_FRAG * 8 + part * 4;       // unit u: 8u channels on
    const bool live = mine && pos < p.positions;
    const int64_t idx_first = (int64_t(img) * p.cout + co_first) * p.howo + rem;
    float dq[U][4], bias[U][4], res[U][4];
    static_for<0, U>([&](auto uc) {
        static_for<0, 4>([&](auto rc) {
            constexpr int u = decltype(uc)::value, r = decltype(rc)::value;
            const int c = min(co_first + 8 * u + r, p.cout - 1);
            dq[u][r] = bias[u][r] = res[u][r] = 0.f;
            if (values) dq[u][r] = p.dq[c];
            if (p.bias) bias[u][r] = p.bias[c];
            if (p.residual) res[u][r] = p.residual[idx_first + int64_t(c - co_first) * p.howo];
        });
    });
    // one consumer scale per tensor or per image; anything else is looked up by element
    const bool q_simple = p.n_qscales == 1 || p.q_group_len == int64_t(p.cout) * p.howo;
    const float q_scale = want_q ? p.q_scales[p.n_qscales == 1 || !q_simple ? 0 : img] : 0.f;

    // ---- K: whole rounds of the ring with the next one requested, then the last round
    typedef int Acc __attribute__((ext_vector_type(R * R / 64)));
    Acc acc[MT];
    static_for<0, MT>([&](auto ic) { acc[decltype(ic)::value] = Acc(0); });
    auto multiply = [&](auto slot) __attribute__((always_inline)) {
        constexpr int s = decltype(slot)::value;
        static_for<0, HALVES>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            static_for<0, MT>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (R == 32) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[s][i][h], b[s][h], acc[i], 0, 0, 0);
                else acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][i][h], b[s][h], acc[i], 0, 0, 0);
            });
        });
    };
    int k = k_first;
    for (int round = 1; round < p.rounds; ++round) {
        static_for<0, D>([&](auto sc) {
            multiply(sc);                                                  // (every wavefront has all steps but the last round's)
            load(sc, k + D);
            ++k;
        });
    }
    static_for<0, D>([&](auto sc) {
        if (k < k_end) multiply(sc);
        ++k;
    });

    // ---- the partial sums meet
    static_for<0, MT>([&](auto ic) {
        static_for<0, PER_FRAG>([&](auto gc) {
            constexpr int i = decltype(ic)::value, g = decltype(gc)::value;
            const v4i sums = {acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
            *reinterpret_cast<v4i *>(lds + (((i * PER_FRAG + g) * W + wave) * 64 + lane) * 16) = sums;
        });
    });
    __syncthreads();
    if (!live) return;
    static_for<0, U>([&](auto uc) {
        constexpr int u = decltype(uc)::value;
        const v4i *from = reinterpret_cast<const v4i *>(lds + ((wave * U + u) * W * 64 + lane) * 16);
        v4i sum = from[0];
        static_for<1, W>([&](auto wc) { sum += from[decltype(wc)::value * 64]; });
        const int left = p.cout - co_first - 8 * u;                        // channels of this unit that exist (4 or more: all)
        const int64_t idx0 = idx_first + int64_t(8 * u) * p.howo;
        auto each = [&](auto &&f) __attribute__((always_inline)) { static_for<0, 4>(f); };
        if (p.out_acc) each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            if (r < left) p.out_acc[idx0 + int64_t(r) * p.howo] = sum[r];
        });
        if (!values) return;
        // one pass per term over the four values, each behind one uniform branch
        float v[4];
        each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fmul_rn(float(sum[r]), dq[u][r]); });
        if (p.bias) each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], bias[u][r]); });
        if (p.residual && !p.res_after) each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], res[u][r]); });
        if (MISHX) each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = mish_value(v[r]); });
        else if (p.act == TSX_ACT_MISH_FAST) each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = mish_short_behind_a_branch(v[r]); });
        else if (p.act != TSX_ACT_NONE) each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            v[r] = apply_act_basic(v[r], p.act, p.slope, idx0 + int64_t(r) * p.howo < p.act_body);
        });
        if (p.residual && p.res_after) each([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __fadd_rn(v[r], res[u][r]); });
        if (p.out_f32) each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            if (r < left) p.out_f32[idx0 + int64_t(r) * p.howo] = v[r];
        });
        if (!want_q) return;
        uint32_t word = 0;
        if (p.n_qscales == 1) each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            word = quantize_pack<r>(__fmul_rn(v[r], q_scale), idx0 + int64_t(r) * p.howo < p.q_bulk8, word);
        });
        else if (q_simple) each([&](auto rc) { constexpr int r = decltype(rc)::value; word = quantize_pack<r>(__fmul_rn(v[r], q_scale), false, word); });
        else each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const int64_t idx = idx0 + int64_t(min(r, left - 1)) * p.howo;
            word = quantize_pack<r>(__fmul_rn(v[r], left > 0 ? p.q_scales[idx / p.q_group_len] : 0.f), false, word);
        });
        word ^= 0x80808080u;
        if (p.out_i8) each([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            if (r < left) p.out_i8[idx0 + int64_t(r) * p.howo] = int8_t(word >> (8 * r));
        });
        if (p.st_out) {
            const int up = p.st_up == 2 ? 2 : 1;
            int8_t *dst = p.st_out + ((int64_t(img) * p.st_hs + up * oh + p.st_pt) * p.st_ws + up * (rem - oh * p.wo) + p.st_pl) * p.st_cp + co_first + 8 * u;
            auto put = [&](int8_t *to) {
                if (left >= 4) *reinterpret_cast<uint32_t *>(to) = word;
                else each([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    if (r < left) to[r] = int8_t(word >> (8 * r));
                });
            };
            put(dst);
            if (up == 2) {
                put(dst + p.st_cp);
                put(dst + int64_t(p.st_ws) * p.st_cp);
                put(dst + int64_t(p.st_ws + 1) * p.st_cp);
            }
        }
    });
}

template <int R, int MT, int D>
int launch(const KsParams &p, hipStream_t stream) {
    const auto kernel = p.act == TSX_ACT_MISH ? conv_i8_ks_kernel<R, MT, D, true> : conv_i8_ks_kernel<R, MT, D, false>;
    constexpr size_t lds_bytes = size_t((R == 32 ? 4 : 1) * MT) * W * 1024;
    static_assert(lds_bytes <= 65536, "what every kernel may have");
    hipLaunchKernelGGL(kernel, dim3(unsigned((p.tiles_m * p.tiles_n + 7) / 8 * 8)), dim3(64 * W), lds_bytes, stream, p);
    TSX_LAUNCH_CHECK("conv_i8_ks_kernel");
    return 0;
}

template <int R, int MT>
int launch_depth(KsParams p, hipStream_t stream) {
    // the ring: the shortest of 1, 2, 3, 5 and 9 K-steps that takes as few rounds as the longest
    constexpr int MOST = R == 16 && MT == 1 ? 9 : 5;
    const int steps = (p.ksteps + W - 1) / W;
    p.rounds = (steps + MOST - 1) / MOST;
    const int depth = (steps + p.rounds - 1) / p.rounds;
    if (depth <= 1) return launch<R, MT, 1>(p, stream);
    if (depth <= 2) return launch<R, MT, 2>(p, stream);
    if (depth <= 3) return launch<R, MT, 3>(p, stream);
    if (depth <= 5) return launch<R, MT, 5>(p, stream);
    return launch<R, MT, MOST>(p, stream);
}

struct KsTile {
    int rows, columns;         // output channels, positions
    int (*launch)(KsParams, hipStream_t);
};
const KsTile TILES[] = {{32, 32, launch_depth<32, 1>}, {16, 16, launch_depth<16, 1>}, {32, 16, launch_depth<16, 2>}};
constexpr int TILE_COUNT = int(sizeof(TILES) / sizeof(TILES[0]));

}  // namespace

void ks_plan(const WsGeom &g, WsPlan *pl) {
    pl->ks = 0;
    if (!pl->ok || g.gemm) return;
    // TSX_CONV_I8_KS, read at every plan: "0" never; a number: that tile wherever the geometry allows (tests).  A test that
    // names the kernel a layer is to take, or those it is not to take, by the other kernels' switches gets what these leave.
    const auto set = [](const char *name) { const char *value = std::getenv(name); return value && value[0]; };
    const char *e = std::getenv("TSX_CONV_I8_KS");
    const int only = e && e[0] ? std::atoi(e) : -1;
    if (only == 0 || only > TILE_COUNT || (only < 0 && (set("TSX_CONV_I8_FLAT") || set("TSX_CONV_I8_RS")))) return;
    const int64_t image = int64_t(g.hs) * g.ws * g.cp, positions = int64_t(g.n) * g.ho * g.wo;
    // 32-bit offsets from a tile's first image
    if (image * (2 + 32 / (int64_t(g.ho) * g.wo)) >= (int64_t(1) << 31) || positions >= (int64_t(1) << 31) - 64) return;
    // Times in us, fitted to 70 layers of 1 to 32 images of 7x7 to 76x76 (residual network and detector shapes): a tile
    // takes 0.25 and what a CU needs to fetch its operands, 59 bytes per ns; the kernels that do not split K take no less
    // than their chain of K-steps.  (One image, us, those kernels -> this one: 3x3 512 to 512 channels 7x7 10.9 -> 5.4, 256
    // to 256 14x14 7.2 -> 4.1, 1x1 1024 to 256 14x14 6.1 -> 3.6, 3x3 100 to 150 13x13 at stride 2 17.8 -> 3.6; 8 images, 3x3
    // 256 to 256 14x14: 7.5, here 8.4.)
    // 1x1 layers with a stride stand against the generic kernel's 128 x 128 tiles, whose epilogue goes element by element where
    // a fragment's 32 channels do not all exist.  (25 images 380 channels 26x130 to 55 at stride 2 with LeakyReLU: 41.4 -> 7.1 us; 4 images 100 100x100 to 90: 15.3 -> 4.3.)
    const int ksteps = g.cblocks * g.kh * g.kw;
    double best = 4.4 + 0.09 * ksteps;
    if (g.kh == 1 && g.kw == 1 && (g.sh > 1 || g.sw > 1))
        best = 5.5 + 0.32 * ksteps + (g.cout % 32 ? 12. * double(ceil_div(ceil_div(positions, 128) * ceil_div(g.cout, 128), 512)) : 0.);
    for (int i = 0; i < TILE_COUNT; ++i) {
        const int64_t tiles = ceil_div(positions, TILES[i].columns) * ceil_div(g.cout, TILES[i].rows);
        if (tiles >= (int64_t(1) << 23)) continue;                         // a launch holds fewer than 2^32 work items
        const double us = 2.9 + double(ceil_div(tiles, 256)) * (0.25 + ksteps * (TILES[i].rows + TILES[i].columns) * 64 / 59e3);
        if (only == i + 1 || (only < 0 && us < best)) {
            best = us;
            pl->ks = i + 1;
        }
    }
}

int ks_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream) {
    if (pl.ks < 1 || pl.ks > TILE_COUNT) return fail(TSX_E_INVALID, "conv_i8_ks: no such tile");
    const KsTile &tile = TILES[pl.ks - 1];
    KsParams p{};
    static_cast<EpiParams &>(p) = ep;
    p.xs = xs;
    p.wp = packed;
    p.cout = g.cout;
    p.frags = pl.coutp / 32;
    p.positions = int(int64_t(g.n) * g.ho * g.wo);
    p.wo = g.wo;
    p.howo = g.ho * g.wo;
    p.hs = g.hs;
    p.ws = g.ws;
    p.cp = g.cp;
    p.sh = g.sh;
    p.sw = g.sw;
    p.kw = g.kw;
    p.taps = g.kh * g.kw;
    p.ksteps = g.cblocks * p.taps;
    p.row_bytes = g.dil_h * g.ws * g.cp;
    p.col_bytes = g.dil_w * g.cp;
    p.cblocks = g.cblocks;
    p.cblocks_magic = div_magic(g.cblocks, p.ksteps);
    p.kw_magic = div_magic(g.kw, p.taps);
    p.tiles_m = int(ceil_div(g.cout, tile.rows));
    p.tiles_n = int(ceil_div(p.positions, tile.columns));
    p.tiles_n_magic = div_magic(p.tiles_n, int64_t(p.tiles_m) * p.tiles_n);
    p.howo_magic = div_magic(p.howo, int64_t(p.positions) + 64);
    p.wo_magic = div_magic(p.wo, p.howo);
    return tile.launch(p, stream);
}

}  // namespace tsx
