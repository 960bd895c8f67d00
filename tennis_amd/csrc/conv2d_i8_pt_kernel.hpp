// The kernel of conv2d_i8_pt.hip; one translation unit per number of K-steps and taps.
#pragma once
#include "conv2d_i8_px_fragment.hpp"

namespace tsx {

struct PtParams : EpiParams {
    const int8_t *xs;      // staged activations [n][hs][ws][cp]
    const int8_t *wp;      // packed weights [ks][coutp/32][2 halves][64 lanes][16]
    int wfrags, rows, ho, wo, hs, ws, cp, sh, sw, kw;
    int th, tw, ctiles, wc, chunks, tap_row, tap_col;       // (tap_row, tap_col: bytes in the window)
    unsigned tw_magic, wc_magic, ho_magic, ctiles_magic, blocks_magic, xs_bytes, st_bytes;
    int tiles, per_xcd, blocks, slots;      // tiles, those of an XCD; workgroups along cout; tiles an XCD works on at a time
};

// wavefronts per SIMD that the registers leave room for
constexpr int pt_waves(int ks, int taps, int fill) { return ks * taps > 9 || fill == 5 ? 2 : 3; }
// fragments of a tile
constexpr int pt_frags(int wn) { return wn == 4 ? 4 : 2; }

// KS: K-steps of 64 channels per tap.  4 / WN wavefronts along cout, each with pt_frags(WN) / WN fragments of a tile.  FILL: 16-byte
// chunks of a window per thread.  MISHX: the activation is the exact Mish.
template <int KS, int TAPS, int WN, int FILL, bool MISHX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(pt_waves(KS, TAPS, FILL)))) void conv_i8_pt_kernel(PtParams p) {
    constexpr int PITCH = KS * 64 + 16, WM = 4 / WN, NF = pt_frags(WN) / WN, STEPS = KS * TAPS;
    __shared__ MishTables mish_tables;
    __shared__ __attribute__((aligned(16))) float terms[4][64];      // each wavefront's scales and biases
    extern __shared__ __attribute__((aligned(16))) int8_t window[];  // [2][pixels][PITCH]
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), half = lane / 32;
    if (MISHX) mish_tables.fill(tid);                                 // (in front of the first barrier)
    const MishTablesInLds tables{&mish_tables};
    // Each XCD takes a contiguous run of tiles with all their channels: halos and cache lines that two tiles share meet in one L2.
    const int xcd = int(blockIdx.x & 7), j = int(blockIdx.x >> 3), slot = udiv(j, p.blocks, p.blocks_magic);
    const int m0 = ((j - slot * p.blocks) * WM + wave % WM) * 32;
    int g = xcd * p.per_xcd + slot;
    const int g_end = min((xcd + 1) * p.per_xcd, p.tiles);
    if (g >= g_end) return;

    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p.xs), 0, int(p.xs_bytes), 0x00020000);
    const auto str = __builtin_amdgcn_make_buffer_rsrc(p.st_out, 0, int(p.st_bytes), 0x00020000);

    // ---- a tile's window: chunk tid + 256 i of 16 bytes at a lane's own offset from the window's first pixel.  What lies behind the last
    // pixel that any output reads comes as zeros.
    const int window_bytes = p.chunks / (4 * KS) * PITCH;
    unsigned fill_off[FILL];
    int fill_dst[FILL];
    static_for<0, FILL>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int q = tid + i * 256, pixel = q / (4 * KS), chunk = q % (4 * KS), wrow = udiv(pixel, p.wc, p.wc_magic);
        fill_off[i] = q < p.chunks ? unsigned(wrow * p.ws + pixel - wrow * p.wc) * unsigned(p.cp) + chunk * 16 : NOWHERE;
        fill_dst[i] = pixel * PITCH + chunk * 16;
    });
    struct Tile { int img, th0, col; };      // image of the first row and that row in it, first column
    auto tile_at = [&](int tile) __attribute__((always_inline)) {
        const int rtile = udiv(tile, p.ctiles, p.ctiles_magic), row = rtile * p.th, img = udiv(row, p.ho, p.ho_magic);
        return Tile{img, row - img * p.ho, (tile - rtile * p.ctiles) * p.tw};
    };
    v4i fill[FILL];
    auto load_window = [&](const Tile &t) __attribute__((always_inline)) {
        // (added up here, saturating: NOWHERE stays beyond the buffer)
        const unsigned at = (unsigned(t.img * p.hs + t.th0 * p.sh) * unsigned(p.ws) + unsigned(t.col * p.sw)) * unsigned(p.cp);
        static_for<0, FILL>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            fill[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, int(__builtin_elementwise_add_sat(fill_off[i], at)), 0, 0));
        });
    };
    auto store_window = [&](int buf) __attribute__((always_inline)) {
        static_for<0, FILL>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if (tid + i * 256 < p.chunks) *reinterpret_cast<v4i *>(window + buf * window_bytes + fill_dst[i]) = fill[i];
        });
    };
    // ---- position l % 32 of this wavefront's fragments: row and column in the tile
    int frow[NF], fcol[NF];
    static_for<0, NF>([&](auto fc) {
        constexpr int f = decltype(fc)::value;
        const int idx = (wave / WM * NF + f) * 32 + lane % 32;
        frow[f] = udiv(idx, p.tw, p.tw_magic);
        fcol[f] = idx - frow[f] * p.tw;
    });
    const int wrap = p.hs - p.ho * p.sh;
    auto where = [&](const Tile &t, int f) __attribute__((always_inline)) {
        PxWhere w;
        const bool over = t.th0 + frow[f] >= p.ho;                    // the next image's
        const int img = t.img + over, oh = t.th0 + frow[f] - (over ? p.ho : 0), ow = t.col + fcol[f];
        const bool ok = frow[f] < p.th && img * p.ho + oh < p.rows && ow < p.wo;
        w.out = NOWHERE;
        w.scale = p.q_scales[p.n_qscales == 1 || !ok ? 0 : img];
        const int up = p.st_up == 2 ? 2 : 1;
        w.st = ok ? unsigned((img * p.st_hs + up * oh + p.st_pt) * p.st_ws + up * ow + p.st_pl) * unsigned(p.st_cp) + m0 + 16 * half : NOWHERE;
        return w;
    };
    const float none[16] = {};                                        // (no residual joins here)
    Tile tile = tile_at(g);
    load_window(tile);
    v4i a[STEPS][2];
    static_for<0, STEPS>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const int8_t *src = p.wp + int64_t(k * p.wfrags + m0 / 32) * 2048 + lane * 16;
        a[k][0] = *reinterpret_cast<const v4i *>(src);
        a[k][1] = *reinterpret_cast<const v4i *>(src + 1024);
    });
    {
        float term = -0.f;               // (a bias that adds nothing)
        if (half == 0) term = p.dq[m0 + lane];
        else if (p.bias) term = p.bias[m0 + lane - 32];
        terms[wave][lane] = term;
    }
    store_window(0);
    lds_barrier();
    int buf = 0;

    auto turn = [&](auto more) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        Tile next = tile;
        if (MORE) {
            next = tile_at(g + p.slots);
            load_window(next);
        }
        static_for<0, NF>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            const PxWhere to = where(tile, f);
            const bool in = frow[f] < p.th;                           // (positions beyond the tile: any pixel of the window)
            const int wrow = in ? frow[f] * p.sh + (tile.th0 + frow[f] >= p.ho ? wrap : 0) : 0;
            const int8_t *b = window + buf * window_bytes + (wrow * p.wc + (in ? fcol[f] : 0) * p.sw) * PITCH + half * 16;
            v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            int at = 0, col = 0;
            static_for<0, TAPS>([&](auto tc) {
                constexpr int tap = decltype(tc)::value;
                static_for<0, KS>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c * TAPS + tap][0], *reinterpret_cast<const v4i *>(b + at + c * 64), acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c * TAPS + tap][1], *reinterpret_cast<const v4i *>(b + at + c * 64 + 32), acc, 0, 0, 0);
                });
                at += p.tap_col;
                if (++col == p.kw) col = 0, at += p.tap_row - p.kw * p.tap_col;
            });
            px_finish<false, false, true, MISHX>(p, acc, terms[wave], none, to, 0, 0, str, str, tables, [] {});
        });
        tile = next;
        if (MORE) {
            store_window(buf ^ 1);
            lds_barrier();
            buf ^= 1;
        }
    };
    for (; g + p.slots < g_end; g += p.slots) turn(std::true_type{});
    turn(std::false_type{});
}

template <int KS, int TAPS, int WN, int FILL, bool MISHX>
int pt_launch_kernel(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream) {
    const auto kernel = conv_i8_pt_kernel<KS, TAPS, WN, FILL, MISHX>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds_bytes, stream, p);
    TSX_LAUNCH_CHECK("conv_i8_pt_kernel");
    return 0;
}

// by kernel: K-steps of 64 channels, taps, fragments side by side, window chunks per thread; each defined by a translation unit
template <int KS, int TAPS, int WN, int FILL>
int pt_launch_layer(const PtParams &p, unsigned grid, size_t lds_bytes, hipStream_t stream);

}  // namespace tsx
