// int8 convolution of layers of six or nine taps on 64 or 128 (padded) input channels that hand out requantized values only, as
// streams of small tiles.
//
// Such a layer is short of work per tile: at 64 channels a fragment of 32 positions x 32 channels is 18 matrix instructions, 576 cycles,
// and its requantization half as many.  The window-stationary kernel keeps these layers busy with setting up: a workgroup per tile
// reads its weights, waits for its window, and works on it at whatever the other workgroups of the CU leave.  Here a
// wavefront holds the weights of its 32 channels in registers (9 K-steps: 72, 18: 144) for all tiles of its workgroup, which are
// small (64 positions, 128 where all four wavefronts share 32 channels): the window of the next one loads into registers while this
// one is multiplied, and waits in the other half of LDS, one barrier a tile.  Windows have a pitch of 80 or 144 bytes a pixel:
// the operands' 16-byte reads are free of bank conflicts.
//
// Measured, us, window-stationary or flat-tile kernel -> here, each layer on buffers of its own.  32 images: 64 to 64 56x56 15.4 -> 11.3, 128 to
// 128 28x28 10.9 -> 10.1 (inside the network 10.7 on both).  8 images: 128 to 256 76x76 25.4 -> 22.1 (1.23 of the 2.3 Pop/s that products
// with both operands' supply alone reach), 64 to 128 304x304 at stride 2 with the exact Mish 45.7 -> 42.0, with the fast one 43.8 -> 32.7; 3x2 taps
// 64 to 64 608x304 at stride 2, 1 with the exact one 70.5 -> 57.8.  300 random layers of 1 to 32 images, 32 to 128 channels: 0.84 of the time in the
// geometric mean, none above 1.05 (with the rules of pt_takes).
//
// Not taken: fp32 values too (a small tile writes pieces of 32 bytes of a plane's rows; 128 to 128 224x224 13.8 -> 17.4); joins (the
// same, and a residual's 16 registers: 128 to 128 76x76 with the exact Mish 30 -> 39).
#include "conv2d_i8_pt.hpp"
#include "conv2d_i8_pt_kernel.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace tsx {

// (defined by the translation units of the kernels)
template <> int pt_launch_layer<1, 9, 1, 3>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 9, 2, 3>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 9, 4, 3>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 9, 1, 5>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 9, 2, 5>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 6, 1, 3>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<1, 6, 2, 3>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<2, 9, 1, 4>(const PtParams &, unsigned, size_t, hipStream_t);
template <> int pt_launch_layer<2, 9, 2, 4>(const PtParams &, unsigned, size_t, hipStream_t);

namespace {

// wavefronts that share 32 channels: the fewest that leave no channels for nobody
int fragments_side_by_side(int cout) { return cout % 128 == 0 ? 1 : cout % 64 == 0 ? 2 : 4; }
// window chunks of 16 bytes per thread of the largest kernel for such layers, 0: none.  They and the weights have to leave room for
// two wavefronts per SIMD.
int most_fill(const WsGeom &g) {
    const int wn = fragments_side_by_side(g.cout), taps = g.kh * g.kw;
    if (g.gemm || g.cout % 32 != 0) return 0;
    if (g.cblocks == 1 && taps == 9) return wn == 4 ? 3 : 5;
    if (g.cblocks == 1 && taps == 6) return wn == 4 ? 0 : 3;
    if (g.cblocks == 2 && taps == 9) return wn == 4 ? 0 : 4;
    return 0;
}

}  // namespace

void pt_plan(const WsGeom &g, WsPlan *pl) {
    // TSX_CONV_I8_PT, read at every plan: "0" never.  A test that names another kernel gets that one.
    const auto set = [](const char *name) { const char *e = std::getenv(name); return e && *e; };
    const char *e = std::getenv("TSX_CONV_I8_PT");
    const int fill = most_fill(g);
    pl->pt = false;
    if (fill == 0 || (e && std::strcmp(e, "0") == 0) || set("TSX_CONV_I8_FLAT") || set("TSX_CONV_I8_RS")) return;
    const int px = 32 * pt_frags(fragments_side_by_side(g.cout)), wrap = g.hs - g.ho * g.sh;
    if (wrap < 0) return;
    const int eh = (g.kh - 1) * g.dil_h + 1, ew = (g.kw - 1) * g.dil_w + 1;
    double best_cost = 0;
    auto consider = [&](int tw) {
        const int th = std::min(px / tw, g.ho), ctiles = int(ceil_div(g.wo, tw)), wc = (tw - 1) * g.sw + ew;
        // (a tile may end in the rows of the next image, which lie `wrap` rows further on)
        const int64_t wpix = (int64_t(th - 1) * g.sh + eh + (g.ho % th ? wrap : 0)) * wc, tiles = ceil_div(int64_t(g.n) * g.ho, th) * ctiles;
        if (wpix * 4 * g.cblocks > fill * 256 || tiles >= (int64_t(1) << 30)) return;
        // a tile's products, and its window's way into LDS
        const double cost = double(tiles) * (px + 0.2 * double(wpix));
        if (pl->pt && cost >= best_cost) return;
        best_cost = cost;
        pl->pt = true;
        pl->pt_th = th;
        pl->pt_tw = tw;
        pl->pt_ctiles = ctiles;
        pl->pt_tiles = tiles;
        pl->pt_wc = wc;
        pl->pt_wpix = int(wpix);
    };
    for (int parts = 1; parts <= 64; ++parts) {
        const int tw = int(ceil_div(g.wo, parts));
        if (tw >= 4 && tw <= px) consider(tw);
    }
    for (int tw = 4; tw <= px; tw *= 2) consider(tw);
    // Tiles that are mostly empty, where windows of strided layers leave little of a map's height and width to choose from: below 0.45 of
    // their positions 1.19 times the other kernels' time (30 layers, 1.64 at most), to 0.6 1.08 (22), above 0.7 0.89 (1240).
    if (pl->pt && int64_t(g.n) * g.ho * g.wo * 5 < pl->pt_tiles * px * 3) pl->pt = false;
    // Too few workgroups leave the tiles that the others could share: 100 to 128 of them 0.91 to 0.97 times as fast as the other
    // kernels (32 images of 14x14, 64 or 128 channels; 7x7 to 512), from 196 on (4 of 28x28 64 to 512; 112x112 64 to 64) 1.06 and more.
    const int wm = 4 / fragments_side_by_side(g.cout);
    if (pl->pt && pl->pt_tiles * (g.cout / 32 / wm) < 160) pl->pt = false;
}

// The workgroups that a CU holds of the kernel that runs the layer, as it is compiled.
static int pt_resident(const WsGeom &g, const WsPlan &pl, bool mishx) {
    const int taps = g.kh * g.kw, fill = pl.pt_wpix * 4 * g.cblocks <= 3 * 256 ? 3 : 5;
    if (!mishx && g.cblocks == 1) return taps == 6 ? 4 : 3;      // (157 registers and fewer, where pt_waves promises two and three)
    return pt_waves(g.cblocks, taps, fill);
}

bool pt_takes(const WsGeom &g, const WsPlan &pl, const EpiParams &ep) {
    if (!pl.pt || ep.residual || ep.out_acc || ep.out_i8 || ep.out_f32 || !ep.st_out) return false;
    // all values in the activation's SIMD body, with one scale per image (or one for all, rounded the same way); tensors that 32-bit
    // offsets reach
    const int64_t image = int64_t(g.cout) * g.ho * g.wo, count = g.n * image, reach = 0xffff0000;
    if (ep.act_body != count || !(ep.n_qscales == 1 ? ep.q_bulk8 == count : ep.q_group_len == image)) return false;
    // What is left to the window-stationary kernel, by the tiles of an XCD times their channel blocks (us, that kernel -> this one).  A little
    // more than its CUs hold two at a time is two turns on a part of them, where that kernel's small tiles fill all: between one round and one
    // and a half, with two channel blocks in and 128 channels out at a time 1.07 in the mean of 47 layers (one image of 151x151 128 to 256 14.1 -> 16.1; 0.92
    // below, 0.91 above), with the exact Mish 1.10 in that of 79 (9 of 70x70 128 to 128 17.5 -> 19.9; 0.92 on both sides); where the flat-tile kernel
    // is the other one 0.96 (84).  The exact Mish makes a turn long: 1.02 in the mean of 136 layers up to 48 (16 of 29x29 64 to 128 8.0 -> 8.4),
    // 0.93 to 64.  It computes empty positions too.
    const bool mishx = ep.act == TSX_ACT_MISH;
    const int wn = fragments_side_by_side(g.cout);
    const int64_t wgs = ceil_div(pl.pt_tiles, 8) * (g.cout / 32 / (4 / wn)), positions = int64_t(g.n) * g.ho * g.wo;
    if (mishx && wn == 1 && wgs <= 48) return false;
    if (mishx && positions * 25 < pl.pt_tiles * 32 * pt_frags(wn) * 18) return false;
    if (!pl.flat && pt_resident(g, pl, mishx) == 2 && (mishx || wn == 1) && wgs > 64 && wgs <= 96) return false;
    return int64_t(g.n) * ep.st_hs * ep.st_ws * ep.st_cp <= reach && int64_t(g.n) * g.hs * g.ws * g.cp <= reach && count < (int64_t(1) << 31);
}

int pt_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream) {
    PtParams p{};
    static_cast<EpiParams &>(p) = ep;
    const int wn = fragments_side_by_side(g.cout), wm = 4 / wn, taps = g.kh * g.kw, pitch = 64 * g.cblocks + 16;
    p.xs = xs;
    p.wp = packed;
    p.wfrags = pl.coutp / 32;
    p.rows = g.n * g.ho;
    p.ho = g.ho;
    p.wo = g.wo;
    p.hs = g.hs;
    p.ws = g.ws;
    p.cp = g.cp;
    p.sh = g.sh;
    p.sw = g.sw;
    p.kw = g.kw;
    p.th = pl.pt_th;
    p.tw = pl.pt_tw;
    p.ctiles = pl.pt_ctiles;
    p.wc = pl.pt_wc;
    p.chunks = pl.pt_wpix * 4 * g.cblocks;
    p.tap_row = g.dil_h * pl.pt_wc * pitch;
    p.tap_col = g.dil_w * pitch;
    p.tw_magic = div_magic(p.tw, 256);
    p.wc_magic = div_magic(p.wc, 2048);
    p.ho_magic = div_magic(p.ho, int64_t(p.rows) + 256);
    p.ctiles_magic = div_magic(p.ctiles, pl.pt_tiles);
    // up to the last pixel that an output reads (the buffer may be a part of a larger one)
    p.xs_bytes = unsigned(((int64_t(g.n - 1) * g.hs + (g.ho - 1) * g.sh + (g.kh - 1) * g.dil_h) * g.ws + (g.wo - 1) * g.sw + (g.kw - 1) * g.dil_w + 1) * g.cp);
    p.st_bytes = unsigned(int64_t(g.n) * ep.st_hs * ep.st_ws * ep.st_cp);
    p.blocks = g.cout / 32 / wm;
    p.tiles = int(pl.pt_tiles);
    p.per_xcd = int(ceil_div(pl.pt_tiles, 8));
    // windows of at most three chunks per thread leave registers for three wavefronts per SIMD
    const bool small = p.chunks <= 3 * 256;
    const int64_t resident = 32 * pt_waves(g.cblocks, taps, small ? 3 : 5);
    // the number of turns with the shortest sequence of rounds; a workgroup's weights and first window take it as long as a turn and a half
    double shortest = 0;
    for (int turns = 16; turns >= 1; --turns) {
        const int64_t slots = ceil_div(p.per_xcd, turns);
        const double time = double(ceil_div(slots * p.blocks, resident)) * (turns + 1.5);
        if (shortest > 0 && time >= shortest) continue;
        shortest = time;
        p.slots = int(slots);
    }
    // ... or one, where CUs hold all workgroups as the kernels are compiled.  (Between what the model takes for that and what it is, us, two turns -> one:
    // 14 images of 73x73 at stride 2 64 to 256 11.4 -> 9.9, 0.89 of the time in the mean of 7 layers; six taps 0.94 in that of 40.)
    if (int64_t(p.per_xcd) * p.blocks <= 32 * pt_resident(g, pl, ep.act == TSX_ACT_MISH)) p.slots = p.per_xcd;
    p.blocks_magic = div_magic(p.blocks, int64_t(p.blocks) * p.slots);
    const unsigned grid = unsigned(8 * p.blocks * p.slots);
    const size_t lds_bytes = size_t(2) * pl.pt_wpix * pitch;
    if (g.cblocks == 2) return wn == 1 ? pt_launch_layer<2, 9, 1, 4>(p, grid, lds_bytes, stream) : pt_launch_layer<2, 9, 2, 4>(p, grid, lds_bytes, stream);
    if (taps == 6) return wn == 1 ? pt_launch_layer<1, 6, 1, 3>(p, grid, lds_bytes, stream) : pt_launch_layer<1, 6, 2, 3>(p, grid, lds_bytes, stream);
    if (wn == 1) return small ? pt_launch_layer<1, 9, 1, 3>(p, grid, lds_bytes, stream) : pt_launch_layer<1, 9, 1, 5>(p, grid, lds_bytes, stream);
    if (wn == 2) return small ? pt_launch_layer<1, 9, 2, 3>(p, grid, lds_bytes, stream) : pt_launch_layer<1, 9, 2, 5>(p, grid, lds_bytes, stream);
    return pt_launch_layer<1, 9, 4, 3>(p, grid, lds_bytes, stream);
}

}  // namespace tsx
