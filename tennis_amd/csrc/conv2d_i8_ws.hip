// Window-stationary int8 convolution (the 3x3 body of ResNet-like nets and config 2; any
// stride, maps of any width through column tiles) on v_mfma_i32_32x32x32_i8
// (the 16x16x64 form runs at half the rate on this part).
//
// Same arithmetic as the generic implicit GEMM in conv2d_i8.hip (exact int32 sums of
// cpu::Conv2DQuantizedCore, src/kernels/cpu/quantized/conv2d_quantized_core.cpp:18-147), but
// a different data movement:
//   * one workgroup (4 wavefronts) owns a tile of TH output rows x TW output columns x 128 output
//     channels; wavefront w owns channels [32w, 32w+32) and all positions of the tile (layers with
//     at most 64 / 32 output channels: 64 / 32 channels, the other wavefronts taking further
//     positions of a 2x / 4x larger tile).  Rows are counted across the whole batch (image n's rows
//     follow image n-1's), so a tile may straddle two images: their staged rows are contiguous in
//     memory, and a position in the second image just reads the window hs - ho*stride rows further
//     down.  Tiles therefore need not divide the image height.  TW is the whole row where the row
//     and its window fit, else a multiple of 32 columns.  A 1x1 layer reading a buffer without halo
//     is tiled as rows of one pixel (the plan's view of the map): any run of consecutive pixels;
//   * per 64-channel block the input *window* that all KH*KW taps of the tile read
//     (((TH-1)*stride + (KH-1)*dil + 1) rows x ((TW-1)*stride + (KW-1)*dil + 1) columns) is copied
//     once into LDS (double buffered, one block ahead, 80-byte pixel stride = bank-conflict-free
//     16-byte reads); every tap is then a shifted read of the same LDS data, so activations cross
//     L2 -> CU once, not KH*KW times, and the K loop needs one barrier per channel block, not per
//     K-step.  A 1x1 layer has one K-step per channel block, too short to cover the window's L2
//     latency one block ahead: its windows hold up to 4 channel blocks per pixel (pixel stride
//     64*blocks + 16) and the blocks of a window are walked like taps;
//   * weights never touch LDS: each wavefront streams its own rows from the packed
//     buffer (1 KiB contiguous per MFMA operand) into a 4-deep register ring, three
//     K-steps ahead of use.
// K order is (channel block, kh, kw); K-steps are padded with zero weights to a multiple
// of the ring depth.
//
// MFMA operand layout (v_mfma_i32_32x32x32_i8): lane l supplies row/column l%32 and the 16
// K bytes of group l/32 (two MFMAs, "halves", cover a 64-byte K-step); accumulator register r
// of lane l is row 8*(r/4) + 4*(l/32) + r%4, column l%32.  Rows = cout, columns = positions.
#include "conv2d_i8_ws_kernel.hpp"
#include "conv2d_i8_ks.hpp"
#include "conv2d_i8_px.hpp"
#include "conv2d_i8_pt.hpp"
#include "tsx_plans.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace tsx {
namespace {

// packed[ks][frag][half][lane][16]: ks = cb*taps + tap; frag = cout/32; lane l: cout frag*32 + l%32,
// channels cb*64 + half*32 + (l/32)*16 + 0..15.  K-steps >= cblocks*taps, rows >= cout, channels >= c: zero.
__global__ __launch_bounds__(256) void ws_pack_kernel(const int8_t *__restrict__ w, int cout, int c, int taps,
                                                     int cblocks, int ksteps_p, int coutp,
                                                     int8_t *__restrict__ packed) {
    const int frags = coutp / 32;
    const int64_t total = int64_t(ksteps_p) * frags * 2 * 64;
    const int64_t id = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const int lane = int(id % 64);
    const int half = int((id / 64) % 2);
    const int frag = int((id / 128) % frags);
    const int ks = int(id / 128 / frags);
    const int cb = ks / taps, tap = ks % taps;
    const int co = frag * 32 + lane % 32;
    const int c0 = cb * 64 + half * 32 + (lane / 32) * 16;
    uint32_t words[4] = {0, 0, 0, 0};
    if (co < cout && cb < cblocks) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int ci = c0 + j;
            const int v = ci < c ? w[(int64_t(co) * c + ci) * taps + tap] : 0;
            words[j / 4] |= uint32_t(v & 0xff) << (8 * (j % 4));
        }
    }
    *reinterpret_cast<uint4 *>(packed + id * 16) = make_uint4(words[0], words[1], words[2], words[3]);
}


}  // namespace

static WsPlan make_ws_plan(const WsGeom &g_in);

WsPlan ws_plan(const WsGeom &g) {
    struct Key {
        WsGeom g;
        PlanSwitch flat, rs, ks, px, pt;
    } key;
    std::memset(&key, 0, sizeof(key));
    key.g = g;
    if (!key.flat.read("TSX_CONV_I8_FLAT") || !key.rs.read("TSX_CONV_I8_RS") || !key.ks.read("TSX_CONV_I8_KS") ||
        !key.px.read("TSX_CONV_I8_PX") || !key.pt.read("TSX_CONV_I8_PT"))
        return make_ws_plan(g);
    return kept_plan<WsPlan>(key, [&] { return make_ws_plan(g); });
}

static WsPlan make_ws_plan(const WsGeom &g_in) {
    WsPlan pl{};
    pl.ok = false;
    // A 1x1 layer reading a buffer without halo is a plain [positions][channels] matrix: rows mean nothing,
    // so it is tiled as rows of ONE pixel (ho*wo of them per image) -- a tile is then any number of
    // consecutive pixels, chosen below as whole fragments whatever the map's width (3136 = 56x56 positions
    // per image give 128-position tiles with no padding; a 608-wide map is no obstacle).
    WsGeom g = g_in;
    if (g.kh == 1 && g.kw == 1 && g.hs == g.ho && g.ws == g.wo && int64_t(g.n) * g.ho * g.wo < (int64_t(1) << 31)) {
        g.ho = g.hs = g_in.ho * g_in.wo;
        g.wo = g.ws = 1;
    }
    pl.ho = g.ho;
    pl.wo = g.wo;
    pl.hs = g.hs;
    pl.ws = g.ws;
    // A tile is TH output rows of the batch-wide row sequence x TW output columns, at most MAX_NT fragments of 32 positions
    // per wavefront.  Candidates are ranked by a model of the busiest CU's time in units of one fragment's work,
    //     (rounds of resident workgroups) x (overlap factor) x (fixed + fragments x slow),
    // where slow = 1.45 for tiles of more than 4 fragments (one workgroup per CU, so one wavefront per SIMD with nothing to
    // hide its LDS/L2 waits).  Ties go to the fewest total fragments (least padding), then to the longest rows.
    constexpr int MAX_NT = 7;
    // few output channels: fewer wavefronts along cout, the others take more positions of a larger tile
    const int wm = g.cout <= 32 ? 1 : g.cout <= 64 ? 2 : 4, wn = 4 / wm;
    const int cap = 32 * MAX_NT * wn;
    if (g.wo < 1 || g.sh < 1 || g.sw < 1) return pl;
    const int wrap = g.hs - g.ho * g.sh;
    const int bm = 32 * WS_FM * wm;
    // GEMM weights are packed once for every kernel that may read them: rows padded to 128
    const int coutp = g.gemm ? (g.cout + 127) / 128 * 128 : (g.cout + bm - 1) / bm * bm;
    const int ksteps_p = (g.cblocks * g.kh * g.kw + RING - 1) / RING * RING;
    double best_cost = -1;
    int64_t best_frags = 0;
    const bool several_taps = g.kh * g.kw > 1;
    auto consider = [&](int tw) {
        const int ctiles = (g.wo + tw - 1) / tw;
        const int wc = (tw - 1) * g.sw + (g.kw - 1) * g.dil_w + 1;
        for (int t = 1; t <= g.ho && t * tw <= cap; ++t) {
            const int nt = ((t * tw + 31) / 32 + wn - 1) / wn;   // fragments per wavefront
            const int64_t tiles = (int64_t(g.n) * g.ho + t - 1) / t * ctiles;
            const bool straddle = g.ho % t != 0;
            const int wr = (t - 1) * g.sh + (g.kh - 1) * g.dil_h + 1 + (straddle && wrap > 0 ? wrap : 0);
            const int wp = wr * wc;
            if (wp > MAX_WP || size_t(2) * wp * PIX > WS_MAX_LDS) continue;   // two windows must fit
            const int64_t wgs = tiles * (coutp / bm);
            const int64_t frags = tiles * nt * wn;
            const int64_t per_cu = (wgs + 255) / 256;
            double cost;
            if (several_taps) {
                // Small near-square tiles: their windows hold few pixels beyond their own, four (one fragment per wavefront)
                // or three (two) of them share a CU, and beyond two rounds a CU takes its next one as soon as one ends.  A
                // wavefront with one fragment still fetches a K-step's weights, 0.3 of a fragment's work at 1.6.  Fitted to
                // some thousand tiles of 35 3x3 layers (us, whole rows before -> now, exact Mish: 8 images of 76x76, 128 to 128
                // channels 25.9 -> 17.8, with a residual 52.8 -> 34.5, 38x38, 256 to 256, with a residual 37.0 -> 25.5, 152x152,
                // 128 to 256 at stride 2, 41.5 -> 31.8; leaky, 76x76, 128 to 256: 26.2 -> 23.0).
                const bool small = nt <= 2 && (wp * 4 + WS_THREADS - 1) / WS_THREADS <= SMALL_FILL;
                const int resident = small ? (nt == 1 ? 4 : 3) : nt <= 4 ? 2 : 1;
                const double rounds = per_cu <= 2 * resident ? double((per_cu + resident - 1) / resident) : double(wgs) / 256 / resident + 0.5;
                const double work = nt * (nt > 4 ? 1.45 : 1.0);
                cost = rounds * (1.0 + 0.55 * double(std::min<int64_t>(per_cu, resident) - 1)) * (0.2 + 0.7 * work + 0.3 * std::max(work, 1.6));
            } else {
                // Workgroups of up to 2 fragments per wavefront fit three to a CU, up to 4 two, larger ones one; those
                // resident together overlap (each further one adds about half of a lone workgroup's time), the rest run in
                // rounds -- so a layer that leaves CUs idle with large tiles takes tiles of half the size.
                const int resident = nt <= 2 ? 3 : nt <= 4 ? 2 : 1;
                const int64_t rounds = (per_cu + resident - 1) / resident;
                cost = double(rounds) * (1.0 + 0.5 * double(std::min<int64_t>(per_cu, resident) - 1)) * (0.5 + nt * (nt > 4 ? 1.45 : 1.0));
            }
            // A 1x1 layer's workgroup is mostly epilogue, its time is the traffic of its tile, and what pays is many small
            // workgroups in flight per CU (us, 32 images, larger tiles -> these: 64 to 256 channels 56x56 with a residual join 63 -> 46,
            // 256 to 128 56x56 20.9 -> 16.9).  The pixel streams write fp32 and staged values of such channels now; of 140
            // layers that they leave, on 192, 320 and more channels or with int8 in planes, this rule and the next change 25: from 0.86 (12 images of 144x144,
            // 256 to 64 with a join, 41.3 -> 35.6) to 1.17 of the model's time (21 of 57x43, 768 to 96, both outputs, 24.1 -> 28.2), 1.03 in the mean.
            if (!several_taps && (!g.gemm || g.cblocks <= 2) && nt > 2) continue;
            // Two fragments share a wavefront's set-up, which pays where every fragment's channels exist and its stores are whole
            // cache lines, that is, where a plane is a multiple of 64 bytes of fp32 (us, one / two: 32 images 256 to 64 56x56 14.5 / 14.0,
            // 128 to 512 28x28 with a join 26.8 / 25.6, 13x48x48, 36 to 256, 15.9 / 14.9; 30 such layers 3 % on average, between
            // -14 % and 7 %).  Elsewhere the model above decides, mostly for one (plane lengths not a multiple of 16: 13x29x226x74 to 52
            // 31.3 / 40.0, 12x8x29x29, 3x3, to 776 23.6 / 27.8; channels not of 32: 24x6x91x91 to 47 24.9 / 33.0, 3x96x122x27 to 801
            // 28.0 / 34.2; 32 channels, a join: 28.7 / 32.0), as for a grid of less than one and a half workgroups per CU (1024 to
            // 256 14x14 9.5 / 10.0).  Only pixels in a row (hs == ho): any tile of them fits.
            if (!several_taps && !g.gemm && g.wo == 1 && g.hs == g.ho && g.ho % 16 == 0 && g.cout % 32 == 0 && wm >= 2 && g.ho >= 64 * wn &&
                nt == (ceil_div(int64_t(g.n) * g.ho, 64 * wn) * (coutp / bm) >= 384 ? 1 : 2)) continue;
            if (best_cost < 0 || cost < best_cost || (cost == best_cost && frags < best_frags)) {
                best_cost = cost;
                best_frags = frags;
                pl.th = t;
                pl.tw = tw;
                pl.ctiles = ctiles;
                pl.nt = nt;
                pl.tiles = tiles;
                pl.wr = wr;
                pl.wc = wc;
                pl.wp = wp;
            }
        }
    };
    if (g.wo <= cap) consider(g.wo);
    if (several_taps) {
        // equal shares of a row, and widths that fill fragments with a few rows
        for (int tw = 64; tw >= 8; tw /= 2)
            if (tw < g.wo) consider(tw);
        for (int parts = 2; parts <= 8; ++parts)
            if ((g.wo + parts - 1) / parts >= 8) consider((g.wo + parts - 1) / parts);
    }
    if (best_cost < 0)
        for (int tw = 32; tw <= cap && tw < g.wo; tw += 32) consider(tw);
    if (best_cost < 0 || pl.tiles >= (int64_t(1) << 31)) return pl;
    pl.wm = wm;
    // 1x1 layers: as many channel blocks per window as divide the layer's, fit the fill registers and LDS
    pl.cbs = 1;
    if (g.kh == 1 && g.kw == 1)
        for (int c = 4; c > 1; c >>= 1)
            if (g.cblocks % c == 0 && pl.wp * 4 * c <= MAX_FILL * WS_THREADS && size_t(2) * pl.wp * (64 * c + 16) <= WS_MAX_LDS) {
                pl.cbs = c;
                break;
            }
    pl.ksteps_p = ksteps_p;
    pl.coutp = coutp;
    pl.packed_bytes = size_t(pl.ksteps_p) * pl.coutp * 64;
    pl.ok = true;
    fl_plan(g_in, &pl);   // layers the flat-tile kernel suits better (same packed weights)
    rs_plan(g_in, &pl);   // ... and the weight-stationary one
    ks_plan(g_in, &pl);   // ... and the one that splits K
    px_plan(g_in, &pl);   // ... and the one for streams of pixels
    pt_plan(g_in, &pl);   // ... and the one for streams of small tiles
    return pl;
}

int ws_pack_weights(const WsGeom &g, const WsPlan &pl, const int8_t *w_oihw, int c, int8_t *packed, hipStream_t stream) {
    const int64_t threads = int64_t(pl.packed_bytes / 16);
    hipLaunchKernelGGL(ws_pack_kernel, dim3(unsigned(ceil_div(threads, 256))), dim3(256), 0, stream, w_oihw, g.cout, c,
                       g.kh * g.kw, g.cblocks, pl.ksteps_p, pl.coutp, packed);
    TSX_LAUNCH_CHECK("ws_pack_kernel");
    return 0;
}

int ws_k_parts(const WsGeom &g, const WsPlan &pl) {
    // One fragment per wavefront, no more workgroups than CUs, and two channel blocks or more for each half of K.  Below 24 K-steps joining the
    // sums takes what halves save: 1x1 layers on 512 to 1024 channels, times without halves : with them 0.97 to 1.025 (1.00 in the mean, 80 layers),
    // on 1536 0.995 to 1.07 (1.02), on 2048 0.99 to 1.10 (1.05).  (Such a launch writes 4 MiB of fp32 at most: never streamed.)
    const int windows = g.cblocks / pl.cbs;
    const size_t lds_bytes = size_t(windows > 1 ? 2 : 1) * pl.wp * (64 * pl.cbs + 16);
    const bool small_fill = ceil_div(pl.wp * 4 * pl.cbs, WS_THREADS) <= SMALL_FILL;
    return pl.nt == 1 && small_fill && pl.tiles * ceil_div(g.cout, 32 * WS_FM * pl.wm) <= 256 && g.cblocks * g.kh * g.kw >= 24 && windows >= 4 &&
           windows % 2 == 0 && 2 * lds_bytes <= 57344 ? 2 : 1;
}

int ws_launch(const WsGeom &g, const WsPlan &plan, const int8_t *xs, const int8_t *packed, const EpiParams &ep,
              hipStream_t stream) {
    WsPlan pl = plan;
    // With the exact Mish a 1x1 layer that hands out its fp32 values evaluates the whole chain for each: tiles of one fragment
    // per wavefront, five wavefronts per SIMD for three: 0.93 of the time in the mean of 70 layers that the pixel streams leave, 0.82 to 1.10
    // (us, 30 images of 59x21, 192 to 128 channels with a join, 28.0 -> 22.8; 9 of 28x44, 640 to 512, 25.3 -> 27.8).  Where only int8
    // leaves, two keep their lead (8 images of 304x304, 64 to 64, 57.6 against 58.4) down to two workgroups per CU.
    if (ep.act == TSX_ACT_MISH && g.kh * g.kw == 1 && pl.wo == 1 && pl.nt == 2 && pl.th == pl.wp && pl.th % 2 == 0 &&
        (ep.out_f32 || pl.tiles * ceil_div(g.cout, 32 * pl.wm) < 512)) {
        pl.nt = 1;
        pl.th = pl.wr = pl.wp = pl.th / 2;
        pl.tiles = ceil_div(int64_t(g.n) * pl.ho, pl.th);
    }
    if (pl.ks) return ks_launch(g, pl, xs, packed, ep, stream);
    if (px_takes(g, pl, ep)) return px_launch(g, pl, xs, packed, ep, stream);
    if (pt_takes(g, pl, ep)) return pt_launch(g, pl, xs, packed, ep, stream);
    if (rs_takes(pl, ep, int64_t(g.n) * g.cout * g.ho * g.wo)) return rs_launch(g, pl, xs, packed, ep, stream);
    if (fl_takes(g, pl, ep)) return fl_launch(g, pl, xs, packed, ep, stream);
    WsParams p{};
    static_cast<EpiParams &>(p) = ep;
    p.xs = xs;
    p.wp = packed;
    p.n = g.n;
    p.cout = g.cout;
    p.coutp = pl.coutp;
    p.ho = pl.ho;   // the plan's view of the map (1-pixel rows for 1x1 layers)
    p.wo = pl.wo;
    p.hs = pl.hs;
    p.ws = pl.ws;
    p.cp = g.cp;
    p.cblocks = g.cblocks;
    p.kh = g.kh;
    p.kw = g.kw;
    p.dil_h = g.dil_h;
    p.dil_w = g.dil_w;
    p.th = pl.th;
    p.wr = pl.wr;
    p.wc = pl.wc;
    p.wpix = pl.wp;
    p.ksteps_p = pl.ksteps_p;
    p.ksteps = g.cblocks * g.kh * g.kw;
    p.wm = pl.wm;
    p.tw = pl.tw;
    p.ctiles = pl.ctiles;
    p.sh = g.sh;
    p.sw = g.sw;
    p.pix = 64 * pl.cbs + 16;
    p.chunk_shift = pl.cbs == 4 ? 4 : pl.cbs == 2 ? 3 : 2;
    p.stage_bytes = 64 * pl.cbs;
    p.tap_row = g.dil_h * pl.wc * p.pix;
    p.tap_col = g.dil_w * p.pix;
    if (pl.cbs > 1) {          // the blocks of a window take the place of taps
        p.cblocks = g.cblocks / pl.cbs;
        p.kh = 1;
        p.kw = pl.cbs;
        p.tap_row = 0;
        p.tap_col = 64;
    }
    p.stream_out = streams_fp32(ep, int64_t(g.n) * g.cout * g.ho * g.wo) ? 1 : 0;
    p.k_parts = ws_k_parts(g, pl);
    p.rowmajor = g.gemm ? 1 : 0;
    if (g.gemm) p.stream_out = 0;
    p.wc_magic = div_magic(p.wc, MAX_WP);
    p.tw_magic = div_magic(p.tw, 4 * 7 * 32);
    p.ow_magic = div_magic(ep.o_w, int64_t(p.ho) * p.wo);
    const int bm = 32 * WS_FM * pl.wm;
    p.tiles = int(pl.tiles);
    p.blocks_m = (g.cout + bm - 1) / bm;
    const int64_t total = pl.tiles * p.blocks_m;
    p.per_xcd = total < (1 << 23) ? int((total + 7) / 8) : 0;      // (a launch holds fewer than 2^32 work items along x)
    p.ho_magic = div_magic(p.ho, int64_t(g.n) * p.ho);
    p.blocks_magic = div_magic(p.blocks_m, total + 7);
    p.ctiles_magic = div_magic(p.ctiles, pl.tiles);
    const dim3 grid = p.per_xcd ? dim3(unsigned(p.per_xcd * 8)) : dim3(unsigned(pl.tiles), unsigned(p.blocks_m));
    // two window buffers (one channel block ahead); a layer whose channels fit one window never swaps and takes one:
    // more workgroups per CU where the window is large (stride-2 3x3 layers on 32 or 64 channels)
    const size_t lds_bytes = size_t(p.cblocks > 1 ? 2 : 1) * pl.wp * (64 * pl.cbs + 16);
    switch (pl.nt) {
        case 1: return ws_launch_nt<1>(p, grid, lds_bytes, stream);
        case 2: return ws_launch_nt<2>(p, grid, lds_bytes, stream);
        case 3: return ws_launch_nt<3>(p, grid, lds_bytes, stream);
        case 4: return ws_launch_nt<4>(p, grid, lds_bytes, stream);
        case 5: return ws_launch_nt<5>(p, grid, lds_bytes, stream);
        case 6: return ws_launch_nt<6>(p, grid, lds_bytes, stream);
        case 7: return ws_launch_nt<7>(p, grid, lds_bytes, stream);
    }
    return fail(TSX_E_INVALID, "conv_i8_ws: unsupported fragment count %d", pl.nt);
}

}  // namespace tsx
