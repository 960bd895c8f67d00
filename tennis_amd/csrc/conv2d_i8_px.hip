// int8 convolution of 1x1 layers, any stride, on 64, 128, 256, 512 or 1024 (padded) input channels, as streams of pixels.
// Same arithmetic, staged input, packed weights and epilogue as conv2d_i8_ws.hip (exact int32 sums of
// cpu::Conv2DQuantizedCore, src/kernels/cpu/quantized/conv2d_quantized_core.cpp:18-147).
//
// Such a layer is mostly epilogue: a fragment of 32 channels x 32 pixels is 2 to 32 MFMAs, and its 16 values a lane some 250
// vector instructions and up to 9 KB of fp32 and int8 values.  What the window-stationary kernel adds to that, a workgroup's set-up
// (some 300 instructions a wavefront) and the chain window - barrier - MFMAs - residual values - stores per tile, is as
// long again.  Here a wavefront keeps the weights of its 32 channels in registers and takes up to three fragments
// one after the other: the pixels of the next one are on their way while one is multiplied and written, its residual
// values from when their registers are free on.  The four wavefronts of a workgroup share their pixels where there are channels for
// that (4 / WN along the output channels, WN fragments side by side).  Pixels go through LDS: read as MFMA operands
// straight from memory, 32 pixels per instruction, they come at 38 bytes per ns and CU from a pitch of 128 bytes on (67 at 64), 16 pixels of
// 64 consecutive bytes at 108.  Scales and biases wait in LDS too, read in every turn: 32 registers less.
//
// us, window-stationary (strided: generic) kernel -> this one, 32 images, each layer on buffers of its own: 64 to 64 channels 56x56 11.0 -> 7.4; 256
// to 64 15.3 -> 11.4; 64 to 256 with a join (fp32 and int8 out) 56.4 -> 52.7, 4.5 TB/s; 128 to 512 28x28 38.5 -> 32.4; 256 to 1024 14x14 24.5 ->
// 21.3 (these read and write fp32 planes in pieces of 128 bytes, for which 205 MB take 37 us at 56x56 and 51 MB 12.4 at 14x14
// with nothing else done; inside the network the first of them stay where they were, 54.2 -> 54.6, 54.3 -> 53.1); 1024 to 256 14x14
// 8.7 -> 7.1; 256 to 512 56x56 at stride 2 22.5 -> 17.7, 1024 to 2048 14x14 20.5 -> 13.2.  8 images with the exact Mish: 64 to 64 304x304, int8 out,
// 57.7 -> 37.2 (vector instructions), fp32 and int8 128 -> 99; 256 to 256 38x38 8.7 -> 6.9.  900 random layers: 0.76 of the time.
#include "conv2d_i8_px.hpp"
#include "conv2d_i8_px_fragment.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace tsx {
namespace {

struct PxParams : EpiParams {
    const int8_t *xs;      // staged activations [n][hs][ws][cp]
    const int8_t *wp;      // packed weights [ks][coutp/32][2 halves][64 lanes][16]
    int cout, wfrags, positions, wo, howo, hs, ws, cp, sh, sw, flat, stream;
    unsigned howo_magic, wo_magic, blocks_magic, out_bytes, st_bytes;
    int groups, per_xcd, blocks, slots;      // groups of WN fragments, those of an XCD; workgroups along cout; groups an XCD works on at a time
};

// Wavefronts per SIMD that the registers have to leave room for, and that the turns are reckoned with.  (Many instantiations fit more
// often as compiled, up to eight times; two K-steps, four fragments side by side and the tables of the exact Mish three times, by their LDS.)
constexpr int px_waves(int ks, int wn, bool res, bool mishx) { return ks == 16 ? 2 : ks == 8 || (res && ks == 4) || (mishx && ks * wn == 8) ? 3 : 4; }

// KS: K-steps of 64 channels.  WN: fragments of a group (4 / WN wavefronts along cout).  RES: a residual joins.  F32, Q: fp32
// values, requantized ones leave.  MISHX: the activation is the exact Mish.  STREAM: the fp32 values in streaming stores.
// PANELS: workgroups by grid.y first (p.blocks of them along cout).
template <int KS, int WN, bool RES, bool F32, bool Q, bool MISHX, bool STREAM = false, bool PANELS = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(px_waves(KS, WN, RES, MISHX)))) void conv_i8_px_kernel(PxParams p) {
    constexpr int PITCH = KS * 64 + 16, CHUNKS = WN * 32 * KS * 4, FILL = (CHUNKS + 255) / 256, WM = 4 / WN;
    __shared__ MishTables mish_tables;
    __shared__ __attribute__((aligned(16))) float terms[4][64];      // each wavefront's scales and biases
    __shared__ __attribute__((aligned(16))) int8_t window[2][WN * 32 * PITCH];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), half = lane / 32;
    if (MISHX) mish_tables.fill(tid);                                 // (in front of the first barrier)
    const MishTablesInLds tables{&mish_tables};
    // Each XCD takes a contiguous run of groups with all their channels: cache lines that two groups share meet in one L2.
    const int xcd = int(blockIdx.x & 7), j = int(blockIdx.x >> 3), slot = udiv(j, p.blocks, p.blocks_magic);
    const int m0 = (((PANELS ? int(blockIdx.y) * p.blocks : 0) + j - slot * p.blocks) * WM + wave % WM) * 32;
    int g = xcd * p.per_xcd + slot;
    const int g_end = min((xcd + 1) * p.per_xcd, p.groups);
    if (g >= g_end) return;

    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p.xs), 0, int(NOWHERE), 0x00020000);
    const auto resr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.residual), 0, int(p.out_bytes), 0x00020000);
    const auto outr = __builtin_amdgcn_make_buffer_rsrc(p.out_f32, 0, int(p.out_bytes), 0x00020000);
    const auto str = __builtin_amdgcn_make_buffer_rsrc(p.st_out, 0, int(p.st_bytes), 0x00020000);

    // ---- a group's pixels: chunk tid + 256 i of 16 bytes, whole pixels one behind the other
    v4i fill[FILL];
    auto load_group = [&](int group) __attribute__((always_inline)) {
        static_for<0, FILL>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int q = tid + i * 256, pixel = q / (4 * KS), chunk = q % (4 * KS);
            const int pos = min(group * (WN * 32) + pixel, p.positions - 1);       // beyond the last: computed, never stored
            unsigned off = unsigned(pos) * unsigned(p.cp) + chunk * 16;
            if (!p.flat) {
                const int img = udiv(pos, p.howo, p.howo_magic), rem = pos - img * p.howo, oh = udiv(rem, p.wo, p.wo_magic);
                off = unsigned((img * p.hs + oh * p.sh) * p.ws + (rem - oh * p.wo) * p.sw) * unsigned(p.cp) + chunk * 16;
            }
            fill[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, int(off), 0, 0));
        });
    };
    auto store_group = [&](int buf) __attribute__((always_inline)) {
        static_for<0, FILL>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int q = tid + i * 256;
            if (i * 256 + 256 <= CHUNKS || q < CHUNKS) *reinterpret_cast<v4i *>(&window[buf][q / (4 * KS) * PITCH + q % (4 * KS) * 16]) = fill[i];
        });
    };
    // ---- position l % 32 of this wavefront's fragment: where its values go
    auto where = [&](int group) __attribute__((always_inline)) {
        PxWhere w;
        const int pos = (group * WN + wave / WM) * 32 + lane % 32, at = min(pos, p.positions - 1);
        const int img = udiv(at, p.howo, p.howo_magic), rem = at - img * p.howo;
        w.out = pos < p.positions ? unsigned((img * p.cout + 4 * half) * p.howo + rem) * 4u : NOWHERE;
        w.scale = 0.f;
        w.st = NOWHERE;
        if (Q) {
            const int oh = udiv(rem, p.wo, p.wo_magic), ow = rem - oh * p.wo;
            w.scale = p.q_scales[p.n_qscales == 1 ? 0 : img];
            const int up = p.st_up == 2 ? 2 : 1;
            if (pos < p.positions) w.st = unsigned((img * p.st_hs + up * oh + p.st_pt) * p.st_ws + up * ow + p.st_pl) * unsigned(p.st_cp) + m0 + 16 * half;
        }
        return w;
    };
    const unsigned row0 = unsigned(m0) * unsigned(p.howo) * 4u, row = unsigned(p.howo) * 4u;
    float res[16];
    auto load_res = [&](const PxWhere &w) __attribute__((always_inline)) {
        if (RES) static_for<0, 16>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            res[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(resr, int(w.out), int(row0 + (8 * (r / 4) + r % 4) * row), 0));
        });
    };
    load_group(g);
    PxWhere now = where(g);
    load_res(now);
    v4i a[KS][2];
    static_for<0, KS>([&](auto kc) {
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
    store_group(0);
    lds_barrier();
    int buf = 0;

    auto turn = [&](auto more) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        PxWhere next = now;
        if (MORE) {
            load_group(g + p.slots);
            next = where(g + p.slots);
        }
        const int8_t *b = &window[buf][(wave / WM * 32 + lane % 32) * PITCH + half * 16];
        v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        static_for<0, KS>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[k][0], *reinterpret_cast<const v4i *>(b + k * 64), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[k][1], *reinterpret_cast<const v4i *>(b + k * 64 + 32), acc, 0, 0, 0);
        });
        px_finish<RES, F32, Q, MISHX, STREAM>(p, acc, terms[wave], res, now, row0, row, outr, str, tables, [&] { if (MORE) load_res(next); });
        now = next;
        if (MORE) {
            store_group(buf ^ 1);
            lds_barrier();
            buf ^= 1;
        }
    };
    for (; g + p.slots < g_end; g += p.slots) turn(std::true_type{});
    turn(std::false_type{});
}

template <int KS, int WN, bool MISHX>
int launch(const PxParams &p, dim3 grid, hipStream_t stream) {
    const bool f32 = p.out_f32, q = p.st_out;
    auto kernel = f32 ? (q ? conv_i8_px_kernel<KS, WN, false, true, true, MISHX> : conv_i8_px_kernel<KS, WN, false, true, false, MISHX>)
                      : conv_i8_px_kernel<KS, WN, false, false, true, MISHX>;
    if (p.stream) kernel = conv_i8_px_kernel<KS, WN, false, true, false, MISHX, true>;
    if constexpr (KS <= 4)
        if (p.residual) kernel = f32 ? (q ? conv_i8_px_kernel<KS, WN, true, true, true, MISHX> : conv_i8_px_kernel<KS, WN, true, true, false, MISHX>)
                                     : conv_i8_px_kernel<KS, WN, true, false, true, MISHX>;
    if constexpr (WN == 1) if (grid.y > 1) {
        kernel = q ? conv_i8_px_kernel<KS, 1, false, true, true, MISHX, false, true> : conv_i8_px_kernel<KS, 1, false, true, false, MISHX, false, true>;
        if constexpr (KS <= 4)
            if (p.residual) kernel = q ? conv_i8_px_kernel<KS, 1, true, true, true, MISHX, false, true> : conv_i8_px_kernel<KS, 1, true, true, false, MISHX, false, true>;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, p);
    TSX_LAUNCH_CHECK("conv_i8_px_kernel");
    return 0;
}

// One turn where an XCD's CUs hold all of its groups, else two or three: more leave the last ones fewer wavefronts to hide their
// memory behind (us for 1, 2, 3, 4, 6 turns: 64 to 256 channels 56x56 with a join 45.6, 46.2, 44.3, 45.9, 46.9; 64 to 64 56x56 7.1, 7.3, 7.0,
// 7.8, 8.8; 64 to 64 304x304 with the exact Mish 46.6, 39.7, 38.7, 39.3, 39.7).  waves: those per SIMD.
int turns_of(int per_xcd, int blocks, int waves) {
    return int(std::min<int64_t>(3, ceil_div(int64_t(per_xcd) * blocks, 32 * waves)));
}
// Weights of 1024 channels leave room for two workgroups per CU: a third on some CUs is a whole turn of nothing beside it, and three
// turns of it were up to a third longer than the best number (us for 1 to 6 turns, 8 images of 40x58, to 384 channels, both outputs, exact Mish, with three by the rule
// above: 35.9, 38.5, 42.4, 35.6, 40.1, 40.6, window-stationary 37.4; 4 of 74x74, to 1024, fp32: 62.8, 58.7, 56.4, 53.4, 53.8, 51.0).  The
// rounds of the busiest CU decide: two that share it take 1.3 of the time of one alone, and before its first turn a workgroup takes
// as long as 1.3 turns, 0.3 of the longer ones with the exact Mish.  131 layers: 0.944 of the time of the rule above and none
// longer than on the window-stationary kernel, where with that rule some took up to 1.13 of its time.
int turns_of_two_per_cu(int per_xcd, int blocks, bool mishx) {
    int best = 1;
    double shortest = 0;
    for (int turns = 1; turns <= 6; ++turns) {
        const int64_t per_cu = ceil_div(ceil_div(per_xcd, turns) * blocks, 32);
        const double time = (turns + (mishx ? 0.3 : 1.3)) * (1.3 * double(per_cu / 2) + double(per_cu % 2));
        if (turns > 1 && time >= shortest) continue;
        shortest = time;
        best = turns;
    }
    return best;
}

template <int KS>
int launch_ks(PxParams &p, hipStream_t stream) {
    const int mfrags = p.cout / 32, wm = mfrags % 4 == 0 ? 4 : mfrags % 2 == 0 ? 2 : 1, wn = 4 / wm;
    p.blocks = mfrags / wm;
    p.groups = int(ceil_div(p.positions, 32 * wn));
    p.per_xcd = int(ceil_div(p.groups, 8));
    const bool mish = p.act == TSX_ACT_MISH;
    const int turns = KS == 16 ? turns_of_two_per_cu(p.per_xcd, p.blocks, mish) : turns_of(p.per_xcd, p.blocks, px_waves(KS, wn, p.residual, mish));
    p.slots = int(ceil_div(p.per_xcd, turns));
    // The workgroups of a group of pixels come one behind the other: they read the same pixels.  Where planes end inside a cache line, the two
    // groups that write a line (and read the residual's) have to meet in L2, and with 16 blocks of channels and more in between the second came
    // when the line had left.  Large outputs of such planes take two blocks at a time (us, window-stationary, all blocks, two: joins of 64 to 2048
    // channels 10 images of 54x54 131.2, 154.5, 118.3, 256 to 4096 32 of 19x19 155, 168, 117; 80 such layers 1.00, 1.18 at most, of the
    // window-stationary kernel's time with all and 0.83 with two).  Smaller outputs stay in L2 (16 blocks, 16 to 32 MiB, 1.00 of the time, up to 1.15),
    // and the exact Mish leaves the second group less behind (32 to 64 MiB 1.01).  In instantiations of their own: the longer way to a workgroup's place, at the head
    // of its chain of loads, cost the other layers 0.5 %.
    const int blocks = p.blocks;
    if (p.out_f32 && !p.stream && p.howo % 32 != 0 && blocks >= 16 && p.out_bytes >= (mish ? 64u << 20 : 32u << 20)) p.blocks = blocks % 2 == 0 ? 2 : 1;
    p.blocks_magic = div_magic(p.blocks, int64_t(p.blocks) * p.slots);
    const dim3 grid(unsigned(8 * p.blocks * p.slots), unsigned(blocks / p.blocks));
    if (wn == 1) return mish ? launch<KS, 1, true>(p, grid, stream) : launch<KS, 1, false>(p, grid, stream);
    if constexpr (KS <= 4) if (wn == 2) return mish ? launch<KS, 2, true>(p, grid, stream) : launch<KS, 2, false>(p, grid, stream);
    if constexpr (KS <= 2) return mish ? launch<KS, 4, true>(p, grid, stream) : launch<KS, 4, false>(p, grid, stream);
    return fail(TSX_E_INVALID, "conv_i8_px: %d channels on %d", p.cout, p.cp);
}

}  // namespace

void px_plan(const WsGeom &g, WsPlan *pl) {
    // TSX_CONV_I8_PX, read at every plan: "0" never
    const char *e = std::getenv("TSX_CONV_I8_PX");
    const int ks = g.cblocks;
    // whole fragments of channels, as many as the kernels compiled for ks have wavefronts along cout
    pl->px = !(e && std::strcmp(e, "0") == 0) && !g.gemm && g.kh == 1 && g.kw == 1 && (ks == 1 || ks == 2 || ks == 4 || ks == 8 || ks == 16) &&
             g.cout % (ks <= 2 ? 32 : ks <= 4 ? 64 : 128) == 0;
}

// with a residual, weights of 512 channels leave too few registers (512 to 2048 7x7, 32 images: 14.0 us window-stationary, 15.5 here)
bool px_joins(const WsGeom &g) { return g.cblocks <= 4; }

bool px_takes(const WsGeom &g, const WsPlan &pl, const EpiParams &ep) {
    if (!pl.px || (ep.residual && !px_joins(g))) return false;
    // fp32 values and staged ones only; all of them in the activation's SIMD body, with one scale per image (or one for all, rounded
    // the same way); tensors that 32-bit offsets reach
    const int64_t image = int64_t(g.cout) * g.ho * g.wo, count = g.n * image, positions = int64_t(g.n) * g.ho * g.wo, reach = 0xffff0000;
    if (ep.out_acc || ep.out_i8 || !(ep.out_f32 || ep.st_out) || ep.act_body != count) return false;
    if (ep.st_out && (int64_t(g.n) * ep.st_hs * ep.st_ws * ep.st_cp > reach || !(ep.n_qscales == 1 ? ep.q_bulk8 == count : ep.q_group_len == image)))
        return false;
    return count * 4 <= reach && int64_t(g.n) * g.hs * g.ws * g.cp <= reach && positions < (int64_t(1) << 31) - 256;
}

int px_launch(const WsGeom &g, const WsPlan &pl, const int8_t *xs, const int8_t *packed, const EpiParams &ep, hipStream_t stream) {
    PxParams p{};
    static_cast<EpiParams &>(p) = ep;
    p.xs = xs;
    p.wp = packed;
    p.cout = g.cout;
    p.wfrags = pl.coutp / 32;
    p.positions = int(int64_t(g.n) * g.ho * g.wo);
    p.wo = g.wo;
    p.howo = g.ho * g.wo;
    p.hs = g.hs;
    p.ws = g.ws;
    p.cp = g.cp;
    p.sh = g.sh;
    p.sw = g.sw;
    p.flat = g.sh == 1 && g.sw == 1 && g.hs == g.ho && g.ws == g.wo;
    p.howo_magic = div_magic(p.howo, p.positions);
    p.wo_magic = div_magic(p.wo, p.howo);
    p.out_bytes = unsigned(int64_t(p.positions) * g.cout * 4);
    p.st_bytes = unsigned(int64_t(g.n) * ep.st_hs * ep.st_ws * ep.st_cp);
    // A large plain fp32 output leaves in streaming stores where planes are whole half cache lines: 137 layers with 64 to 1024 channels
    // 0.93 of the time of stores that L2 keeps (us, window-stationary, L2, streaming: 7 images of 32x32 1024 to 2048 30.8, 35.0, 28.6;
    // 26 of 200x200 128 to 64 71.6, 85.7, 65.2), and what the kernels behind it read stays in L2 (the ResNet-50 shape on 32 images: its
    // first projection 22.3 -> 23.0, the join behind it 55.0 -> 44.8).  Planes of another length write parts of lines, which L2 joins.
    p.stream = streams_fp32(ep, int64_t(p.positions) * g.cout) && p.howo % 16 == 0;
    switch (g.cblocks) {
        case 1: return launch_ks<1>(p, stream);
        case 2: return launch_ks<2>(p, stream);
        case 4: return launch_ks<4>(p, stream);
        case 8: return launch_ks<8>(p, stream);
        case 16: return launch_ks<16>(p, stream);
    }
    return fail(TSX_E_INVALID, "conv_i8_px: %d channel blocks", g.cblocks);
}

}  // namespace tsx
