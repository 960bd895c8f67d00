// Staging by runs of a channel plane: the transposition from [channel][pixel] to [pixel][channel] through LDS.
//
// Bound by memory: 4 (or 1) bytes read and 1 written per element.  A channel plane of an image is one contiguous run of
// h*w elements whatever its width, so a workgroup takes 4 x 64 consecutive pixels of it, not a row: wavefront k the 16
// channels of chunk k, a lane four consecutive pixels -- one 16-byte load (4-byte for int8 sources) per channel at the
// element's own alignment, all 16 of a lane in flight at once, 1 KiB contiguous per load instruction.  The last lane of
// a plane takes its last four pixels again instead of a masked remainder.  Quantized bytes are packed by the
// conversion instruction, four int8 channels by byte permutes; the tile goes through LDS so that a pixel's 64 channels
// leave as one 64-byte run.  Halo pixels are written by workgroups of their own behind the others of the launch.
//
// Rows of one staged row per workgroup (loads as wide as the row's length allows, one byte or float for odd widths, few
// workgroups on small maps) took 87 us for 6x493x49x205 int8 and 63 us for 25x380x26x130, one lane per 16-byte chunk of
// a wide row 159 us for 17x176x85x281 fp32 (0.36 GB); this form 12, 12 and 68 (5.3 TB/s), and 8.6 instead of 9.1 on
// 32x256x28x28 fp32 (33 MB: one round of workgroups, so latency).
#include "stage_i8.hpp"
#include "igemm_i8.hpp"

#include <algorithm>

namespace tsx {
namespace {

typedef float v4f_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_a1 __attribute__((aligned(1)));

constexpr int SP_POS = 256;                              // pixels of a workgroup
constexpr int SP_PIX = 80;                               // LDS bytes per pixel (64 + 16), 16 more per four pixels:
constexpr int SP_LDS = SP_POS * SP_PIX + SP_POS / 4 * 16;    // a lane's writes are then spread over all banks

__device__ __forceinline__ int sp_addr(int t) { return t * SP_PIX + (t >> 2) * 16; }

struct StagePlanes {
    StageGeom g;
    const void *src;
    const float *scales;
    int n_scales;
    int64_t group_len, bulk8;
    int8_t *xs;
    int hw, groups;                 // pixels of a plane, groups of four of them
    int gblocks, gper;              // workgroups along the plane, groups each takes
    int cblocks;                    // blocks of 64 channels
    unsigned interior, per_xcd;     // workgroups of pixels, of them per XCD
    int hr, wc;                     // rows and columns of the map that are staged
    int halo_px;                    // halo pixels per image
    int64_t halo_chunks;            // 16-byte chunks of them in all
    unsigned w_magic;
};

// The halo: T(padding_value) in the real channels, 0 in the channel padding.
__device__ __forceinline__ void stage_halo_chunk(const StagePlanes &p, int64_t id) {
    const StageGeom &g = p.g;
    const int cpc = g.cp / 16;
    const int64_t hp_all = id / cpc;
    const int chunk = int(id - hp_all * cpc);
    const int img = int(hp_all / p.halo_px);
    int hp = int(hp_all - int64_t(img) * p.halo_px);
    int row, col;
    const int above = min(g.pad_top, g.hs) * g.ws, below = (g.hs - min(g.pad_top, g.hs) - p.hr) * g.ws;
    if (hp < above + below) {
        row = hp / g.ws;
        col = hp - row * g.ws;
        if (hp >= above) row += p.hr;
    } else {
        hp -= above + below;
        const int side = g.ws - p.wc;                          // halo pixels beside one interior row
        row = hp / side;
        const int k = hp - row * side;
        row += g.pad_top;
        col = k < g.pad_left ? k : p.wc + k;
    }
    uint32_t words[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int real = min(max(g.c - (chunk * 16 + v * 4), 0), 4);
        words[v] = real == 0 ? 0u : (uint32_t(g.pad_value & 0xff) * 0x01010101u) & (0xffffffffu >> (8 * (4 - real)));
    }
    *reinterpret_cast<uint4 *>(p.xs + ((int64_t(img) * g.hs + row) * g.ws + col) * g.cp + chunk * 16) =
        make_uint4(words[0], words[1], words[2], words[3]);
}

// words[pixel][channel / 4] := the quantized elements of 16 channels x 4 pixels.  EVEN: round half to even; MIXED: each
// element chooses its scale and rounding by its index relative to the first plane (StageBounds).
struct StageBounds {
    float s_prev, s_next;     // scales in front of element lo / from element hi on
    int lo, hi, body;         // elements in front of `body` round half to even
    int hw, pos;
};
template <bool EVEN, bool MIXED>
__device__ __forceinline__ void stage_pack(const float (&v)[16][4], float s, const StageBounds &b, uint32_t (&words)[4][4]) {
    static_for<0, 16>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        static_for<0, 4>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const int o = MIXED ? i * b.hw + b.pos + j : 0;
            const float sc = MIXED ? (o < b.lo ? b.s_prev : o >= b.hi ? b.s_next : s) : s;
            words[j][i / 4] = quantize_pack<i % 4>(__fmul_rn(v[i][j], sc), MIXED ? o < b.body : EVEN, words[j][i / 4]);
        });
    });
}

template <bool QUANT>
__global__ __launch_bounds__(256) void stage_planes_kernel(StagePlanes p) {
    __shared__ __attribute__((aligned(16))) int8_t tile[SP_LDS];
    const StageGeom &g = p.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (blockIdx.x >= p.per_xcd * 8) {
        const int64_t id = int64_t(blockIdx.x - p.per_xcd * 8) * 256 + tid;
        if (id < p.halo_chunks) stage_halo_chunk(p, id);
        return;
    }
    // Workgroups are dealt round-robin to the 8 XCDs, each with its own L2: give each XCD a contiguous run of them, so
    // that the cache lines neighbours share -- the ends of a run of pixels, a pixel's other channels -- meet in one L2
    const unsigned b = (blockIdx.x % 8) * p.per_xcd + blockIdx.x / 8;
    if (b >= p.interior) return;
    const int cb = b % p.cblocks;
    const unsigned rest = b / p.cblocks;
    const int gb = rest % p.gblocks, ni = rest / p.gblocks;
    const int g0 = gb * p.gper, gn = min(p.gper, p.groups - g0);
    const int c0 = cb * 64 + wave * 16;                       // first channel of this wavefront
    const int creal = min(max(g.c - c0, 0), 16);              // of its 16, those that exist
    const int pos = min(4 * (g0 + min(lane, gn - 1)), p.hw - 4);
    uint32_t words[4][4];                                     // [pixel][channel quad]
    static_for<0, 16>([&](auto i) { words[decltype(i)::value / 4][decltype(i)::value % 4] = 0u; });
    if (creal > 0) {
        const int64_t plane0 = (int64_t(ni) * g.c + c0) * p.hw;   // linear index of the first channel's plane
        const int64_t last = plane0 + int64_t(creal) * p.hw - 1;
        if constexpr (QUANT) {
            float v[16][4];
            static_for<0, 16>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                const v4f_a4 t = *reinterpret_cast<const v4f_a4 *>(static_cast<const float *>(p.src) + plane0 + int64_t(min(i, creal - 1)) * p.hw + pos);
                v[i][0] = t[0];
                v[i][1] = t[1];
                v[i][2] = t[2];
                v[i][3] = t[3];
            });
            // one scale and one way of rounding for all of the wavefront's elements, or a choice per element where a
            // scale group (the reference's group length is a rounded quotient) or the body of its SIMD loop ends
            const bool even = p.n_scales == 1 && last < p.bulk8;
            const int64_t group0 = ni * p.group_len;
            const bool one_scale = p.n_scales == 1 || (plane0 >= group0 && last < group0 + p.group_len);
            const int si = p.n_scales == 1 ? 0 : ni;
            const float s = p.scales[si];
            if (one_scale && (even || p.n_scales > 1 || plane0 >= p.bulk8)) {
                const StageBounds none{};
                if (even) stage_pack<true, false>(v, s, none, words);
                else stage_pack<false, false>(v, s, none, words);
            } else {
                // elements in front of `lo` belong to the group before, from `hi` on to the next; those in front of `body`
                // round to even (all relative to the first plane; 16 planes are fewer than 2^31 elements)
                auto rel = [&](int64_t e) { return int(min(max(e - plane0, int64_t(0)), int64_t(0x7fffffff))); };
                const bool one = p.n_scales == 1;
                const StageBounds bounds{p.scales[max(si - 1, 0)], p.scales[min(si + 1, p.n_scales - 1)], one ? 0 : rel(group0),
                                         one ? 0x7fffffff : rel(group0 + p.group_len), one ? rel(p.bulk8) : 0, p.hw, pos};
                stage_pack<false, true>(v, s, bounds, words);
            }
            static_for<0, 16>([&](auto i) { words[decltype(i)::value / 4][decltype(i)::value % 4] ^= 0x80808080u; });
        } else {
            uint32_t v[16];
            static_for<0, 16>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                v[i] = *reinterpret_cast<const u32_a1 *>(static_cast<const int8_t *>(p.src) + plane0 + int64_t(min(i, creal - 1)) * p.hw + pos);
            });
            // 4 x 4 bytes: [channel][pixel] -> [pixel][channel]
            static_for<0, 4>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                const uint32_t lo01 = __builtin_amdgcn_perm(v[4 * q + 1], v[4 * q], 0x05010400u), hi01 = __builtin_amdgcn_perm(v[4 * q + 1], v[4 * q], 0x07030602u);
                const uint32_t lo23 = __builtin_amdgcn_perm(v[4 * q + 3], v[4 * q + 2], 0x05010400u), hi23 = __builtin_amdgcn_perm(v[4 * q + 3], v[4 * q + 2], 0x07030602u);
                words[0][q] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
                words[1][q] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
                words[2][q] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
                words[3][q] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
            });
        }
        if (creal < 16) static_for<0, 4>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            const int real = min(max(creal - 4 * q, 0), 4);
            const uint32_t keep = real == 0 ? 0u : 0xffffffffu >> (8 * (4 - real));
            static_for<0, 4>([&](auto jc) { words[decltype(jc)::value][q] &= keep; });
        });
    }
    if (lane < gn) static_for<0, 4>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const v4i chunk = {int(words[j][0]), int(words[j][1]), int(words[j][2]), int(words[j][3])};
        *reinterpret_cast<v4i *>(&tile[sp_addr(lane * 4 + j) + wave * 16]) = chunk;
    });
    __syncthreads();
    // four lanes write a pixel's 64 channels
    static_for<0, 4>([&](auto ic) {
        const int t = decltype(ic)::value * 64 + (tid >> 2);
        const int f = min(4 * (g0 + (t >> 2)), p.hw - 4) + (t & 3);
        const int hi = udiv(f, g.w, p.w_magic), wi = f - hi * g.w;
        if ((t >> 2) < gn && hi < p.hr && wi < p.wc)
            *reinterpret_cast<v4i *>(p.xs + ((int64_t(ni) * g.hs + hi + g.pad_top) * g.ws + wi + g.pad_left) * g.cp + cb * 64 + (tid & 3) * 16) =
                *reinterpret_cast<const v4i *>(&tile[sp_addr(t) + (tid & 3) * 16]);
    });
}

}  // namespace

bool stage_planes_takes(const StageGeom &g) {
    const int64_t hw = int64_t(g.h) * g.w;
    return hw >= 4 && hw < (int64_t(1) << 27) && g.cp % 64 == 0 && g.cp >= g.c;
}

int stage_planes(const StageGeom &g, const void *src, const float *scales, int n_scales, int64_t group_len, int64_t bulk8, int8_t *xs,
                 hipStream_t stream) {
    StagePlanes p{};
    p.g = g;
    p.src = src;
    p.scales = scales;
    p.n_scales = n_scales;
    p.group_len = group_len;
    p.bulk8 = bulk8;
    p.xs = xs;
    p.hw = g.h * g.w;
    p.groups = (p.hw + 3) / 4;
    p.gblocks = (p.groups + SP_POS / 4 - 1) / (SP_POS / 4);
    p.gper = (p.groups + p.gblocks - 1) / p.gblocks;       // no nearly empty last workgroup
    p.cblocks = g.cp / 64;
    const int64_t interior = int64_t(g.n) * p.gblocks * p.cblocks;
    p.hr = std::max(0, std::min(g.h, g.hs - g.pad_top));
    p.wc = std::max(0, std::min(g.w, g.ws - g.pad_left));
    if (p.hr == 0 || p.wc == 0) p.hr = p.wc = 0;
    p.halo_px = g.hs * g.ws - p.hr * p.wc;
    p.halo_chunks = int64_t(g.n) * p.halo_px * (g.cp / 16);
    p.w_magic = div_magic(g.w, p.hw);
    const int64_t per_xcd = (interior + 7) / 8, blocks = per_xcd * 8 + (p.halo_chunks + 255) / 256;
    TSX_REQUIRE(blocks < (int64_t(1) << 31), "stage: too many pixels for one launch");
    p.interior = unsigned(interior);
    p.per_xcd = unsigned(per_xcd);
    if (scales) hipLaunchKernelGGL(stage_planes_kernel<true>, dim3(unsigned(blocks)), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(stage_planes_kernel<false>, dim3(unsigned(blocks)), dim3(256), 0, stream, p);
    TSX_LAUNCH_CHECK("stage_planes_kernel");
    return 0;
}

}  // namespace tsx
