// Shared host/device helpers of the gfx950 kernels behind include/tsx_hip.h.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <type_traits>

#include "tsx_hip.h"
#include "tsx_mish.hpp"

namespace tsx {

// Thread-local message behind tsx_last_error().
char *error_buffer();
int fail(int code, const char *fmt, ...);

inline int check_hip(hipError_t e, const char *what) {
    if (e == hipSuccess) return 0;
    return fail(int(e), "%s: %s", what, hipGetErrorString(e));
}

#define TSX_HIP(expr)                                        \
    do {                                                     \
        int _rc = ::tsx::check_hip((expr), #expr);           \
        if (_rc) return _rc;                                 \
    } while (0)

#define TSX_REQUIRE(cond, ...)                               \
    do {                                                     \
        if (!(cond)) return ::tsx::fail(TSX_E_INVALID, __VA_ARGS__); \
    } while (0)

// Launch check: the reference checks the runtime right after every launch and ejects
// (include/kernels/gpu/gpu_kernel.h:13-19); here the error code goes back over the C ABI.
#define TSX_LAUNCH_CHECK(name) TSX_HIP(hipGetLastError())

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline int64_t round_up(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

// Output extent of a convolution (include/backend/common_function.h:30-40).
inline int conv_out(int in, int pad_a, int pad_b, int k, int stride, int dilation) {
    return (in + pad_a + pad_b - (dilation * (k - 1) + 1)) / stride + 1;
}

// ---------------------------------------------------------------------------
// Device-side scalar semantics shared by the quantize kernel and fused epilogues.
// ---------------------------------------------------------------------------
#ifdef __HIPCC__

// Compile-time loop: register arrays are only ever indexed by constants, which keeps them
// in VGPRs (loop-indexed arrays, and arrays of HIP's uint4/float4 structs, can end up in
// scratch memory).
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// q = clamp(round(v), -128, 127) with the reference's x86 conversion behaviour:
// NaN and |v| >= 2^31 convert to INT_MIN, i.e. -128 after the clamp
// (src/kernels/cpu/quantize.cpp:15-29,83-96).
__device__ __forceinline__ int quantize_value(float v, bool half_even) {
    // rintf = round half to even (_mm256_cvtps_epi32).  round() = half away from zero, computed as
    // trunc(v + copysign(0.5 - 2^-25, v)): the addend is the float below 0.5, so 0.49999997 stays 0 while
    // every x.5 still reaches the next integer (the sum rounds up to it); equal to roundf(v) for
    // |v| < 2^23 and, like it, far outside the clamp beyond (three instructions instead of roundf's six;
    // this runs once per element in the staging kernel, which is bound by its arithmetic).
    const float away = __builtin_truncf(v + __builtin_copysignf(0.49999997f, v));
    const float r = half_even ? __builtin_rintf(v) : away;
    // selects, not branches: this runs once per output element in the epilogues
    const float c = __builtin_amdgcn_fmed3f(r, -128.f, 127.f);   // the clamp as one instruction; NaN is overridden below
    const bool in_range = __builtin_fabsf(v) < 2147483648.0f;   // false for NaN as well
    return in_range ? int(c) : -128;
}

// Byte SEL of `word` := quantize_value(v, half_even) + 128 (offset binary; the caller XORs the finished word with
// 0x80808080): the conversion instruction saturates to [0, 255] and packs, so clamp, conversion and packing are one
// instruction.  r + 128 is exact wherever the clamp does not apply anyway; NaN and |v| >= 2^31 give byte 0 = -128, the
// reference's INT_MIN after its clamp, as in quantize_value.
template <int SEL>
__device__ __forceinline__ uint32_t quantize_pack(float v, bool half_even, uint32_t word) {
    const float away = __builtin_truncf(v + __builtin_copysignf(0.49999997f, v));
    const float r = half_even ? __builtin_rintf(v) : away;
    const bool in_range = __builtin_fabsf(v) < 2147483648.0f;   // false for NaN as well
    return __builtin_amdgcn_cvt_pk_u8_f32(in_range ? __fadd_rn(r, 128.f) : 0.f, SEL, word);
}

// relu / leaky_relu of element `in_body` (= linear index < 4*floor(count/4) of the whole
// tensor): SIMD body vs scalar tail of src/kernels/cpu/relu.cpp:30-52 and
// leaky_relu.cpp:41-66.  Body: max(x,0) returns +0 for -0 and NaN; the leaky form is one
// fused multiply-add in the reference's FMA build.  Tail: std::max / ternary.
// none / relu / leaky_relu only: for kernels that unroll the call many times -- the Mish branch below is a few hundred
// instructions (double-precision log), and dozens of inlined copies of it put the taken branches of the cheap
// activations an instruction-cache miss apart.
__device__ __forceinline__ float apply_act_basic(float v, int act, float slope, bool in_body) {
    if (act == TSX_ACT_RELU) {
        return in_body ? (v > 0.f ? v : 0.f) : (v < 0.f ? 0.f : v);
    }
    if (act == TSX_ACT_LEAKY_RELU) {
        if (in_body) {
            const float mx = v > 0.f ? v : 0.f;
            const float mn = v < 0.f ? v : 0.f;
            return __builtin_fmaf(slope, mn, mx);
        }
        return v > 0.f ? v : __fmul_rn(v, slope);
    }
    return v;
}

// Mish, softplus and tanh in the host's arithmetic: tsx_mish.hpp (shared with the CPU build that pins them)
// The fast form for layers bound by the activation's arithmetic (the 608x608 and 304x304 layers of a YOLOv4-shaped
// backbone spend more issue slots on an exact Mish than the VALUs have in the time the layer's bytes take): one
// exponential and one reciprocal at the hardware's 1 ulp,
//     tanh(softplus(x)) = 1 - 2 / (w + 2),  w = e (e + 2),  e = e^x = 2^(x log2 e),
// with -2 / (w + 2) as the reciprocal of -(e (e/2 + 1) + 1): five operations and the two transcendental ones (an issue slot
// of four cycles and ten cycles each).  1 - 2r with r = 1 / (w + 2) in (0, 0.5] has the shape of the host's tanh: an absolute
// error of about 1e-7 in the quotient, so about 1e-7 |x| in the result (at most 2e-6 absolute for negative x, where Mish
// itself is small) -- and, like the host's, exactly 0 (-0 for the product) once x is below about -17, where the divisor
// rounds to 1; 1 above 17, also where e^x or its square overflow.
// NaN -> NaN, +-inf as the host's.  A requantized int8 value differs from the exact form's in about one of a million.
// Opt-in (TSX_ACT_MISH_FAST); TSX_ACT_MISH is the exact form, mish_value.
__device__ __forceinline__ float mish_minus_quotient(float x) {      // -2 / (w + 2)
    const float e = __builtin_amdgcn_exp2f(__fmul_rn(x, 1.4426950216293335f));
    return __builtin_amdgcn_rcpf(__builtin_fmaf(e, __builtin_fmaf(e, -0.5f, -1.f), -1.f));
}
__device__ __forceinline__ float mish_short(float x) {
    return __fmul_rn(x, __fadd_rn(1.f, mish_minus_quotient(x)));
}

// quantize_pack for N values, N / 4 words of four int8 each (not offset binary), in 5.25 instructions an element for 7: the
// clamp by the median of three (a NaN gives its lower end), the rounding offset, a conversion that truncates, and three byte
// operations a word; one look at the largest of the N finds what converts to INT_MIN, products of 2^31 and more.  With
// activate_results, of a fragment's 29 instructions a value 11 went; the kernels wait for memory more than they issue, so
// it is little: the ResNet-50 shape on 32 images 1013 -> 1001 us, 64 to 64 channels 56x56 8.9 -> 8.5.
template <int N>
__device__ __forceinline__ void quantize_words(const float (&v)[N], float scale, bool half_even, uint32_t (&word)[N / 4]) {
    float t[N];
    static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; t[r] = __fmul_rn(v[r], scale); });
    float top = t[0];
    static_for<0, N / 2>([&](auto rc) { constexpr int r = decltype(rc)::value; top = __builtin_fmaxf(__builtin_fmaxf(top, t[2 * r]), t[2 * r + 1]); });
    if (top >= 2147483648.0f)
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; t[r] = t[r] >= 2147483648.0f ? -128.f : t[r]; });
    static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; t[r] = __builtin_amdgcn_fmed3f(t[r], -128.f, 127.f); });
    if (half_even) static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; t[r] = __builtin_rintf(t[r]); });
    else static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; t[r] += __builtin_copysignf(0.49999997f, t[r]); });
    static_for<0, N / 4>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        word[g] = __builtin_amdgcn_perm(unsigned(int(t[4 * g + 1])), unsigned(int(t[4 * g])), 0x0c0c0400u) |
                  __builtin_amdgcn_perm(unsigned(int(t[4 * g + 3])), unsigned(int(t[4 * g + 2])), 0x04000c0cu);
    });
}

// N values of a fragment, results of arithmetic (no signaling NaN) in the activations' SIMD body, whose ReLU and LeakyReLU the
// hardware's maximum and minimum are: a NaN, and a zero of either sign, give +0.  As instructions, since the compiler first
// quiets what it cannot tell from a signaling NaN.  The empty statement holds the fast Mish behind its branch: without a
// side effect there the compiler computed it for every value in front of the test of the activation, in every layer of these
// kernels (16 exponentials, 16 reciprocals and 96 other instructions a fragment).
__device__ __forceinline__ float max_zero(float v) {
    float r;
    asm("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ float min_zero(float v) {
    float r;
    asm("v_min_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}
template <int N>
__device__ __forceinline__ void activate_results(float (&v)[N], int act, float slope) {
    if (act == TSX_ACT_RELU) {
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = max_zero(v[r]); });
    } else if (act == TSX_ACT_LEAKY_RELU) {
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = __builtin_fmaf(slope, min_zero(v[r]), max_zero(v[r])); });
    } else if (act == TSX_ACT_MISH_FAST) {
        asm volatile("; fast Mish");
        static_for<0, N>([&](auto rc) { constexpr int r = decltype(rc)::value; v[r] = mish_short(v[r]); });
    }
}
// ... for a single value, likewise not to be computed in front of the branch that it stands behind
__device__ __forceinline__ float mish_short_behind_a_branch(float v) {
    asm volatile("; fast Mish");
    return mish_short(v);
}

// The activation of every epilogue: none / relu / leaky_relu / Mish (exact) / Mish (fast), an element at a time; activate_results is
// the same for a whole fragment of the SIMD body.  Both give the same bits for every value, so an element's value never depends on the
// kernel or tile it falls into, and a fused node gives what the separate operators give.
__device__ __forceinline__ float apply_act(float v, int act, float slope, bool in_body) {
    if (act == TSX_ACT_MISH) return mish_value(v);
    if (act == TSX_ACT_MISH_FAST) return mish_short_behind_a_branch(v);
    return apply_act_basic(v, act, slope, in_body);
}
// The tables of the exact Mish in the workgroup's LDS: the 32 entries of the exponential's take two banks each, so a read of
// any 64 of them is free of conflicts; the logarithm's two are read by one instruction, at multiples of 512 bytes from each other.
// (Held in the wavefront's lanes and read with ds_bpermute, a look-up takes 28 cycles of a SIMD's share of the LDS pipe per 32
// bits: seven of them were as long as the arithmetic.)
struct __attribute__((aligned(512))) MishTables {
    double twice_inverse[256], log_of[256];
    uint64_t exp2[32];
    __device__ __forceinline__ void fill(int tid) {       // by at least 256 threads, in front of a barrier
        if (tid >= 256) return;
        const MishTablesInMemory from;
        twice_inverse[tid] = from.twice_inverse(tid);
        log_of[tid] = from.log_of(tid);
        if (tid < 32) exp2[tid] = from.exp2(tid);
    }
};
struct MishTablesInLds {
    const MishTables *t;
    __device__ __forceinline__ uint64_t exp2(uint32_t i) const { return t->exp2[i]; }
    __device__ __forceinline__ double twice_inverse(int i) const { return t->twice_inverse[i]; }
    __device__ __forceinline__ double log_of(int i) const { return t->log_of[i]; }
};

// The exact Mish of the 16 values of an accumulator fragment, two values per turn of a loop that stays a loop: each
// value's chain holds a dozen double-precision temporaries and twenty constants, and sixteen chains unrolled side by
// side would push a kernel that keeps its accumulators and operands in registers into scratch memory; two give the
// scheduler something to put into the other's latencies.  The loop counter is uniform: the values are reached by
// register indexing.
template <class Table>
__device__ __forceinline__ void mish_fragment(float (&v)[16], const Table &table) {
    typedef float v16f __attribute__((ext_vector_type(16)));
    v16f t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = v[r];
    MishAddends add;
    asm volatile("" : "+v"(add.exp2), "+v"(add.log));
#pragma clang loop unroll(disable)
    for (int r = 0; r < 16; r += 2) {
        const float a = mish_value(t[r], table, add), b = mish_value(t[r + 1], table, add);
        t[r] = a;
        t[r + 1] = b;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = t[r];
}

// The exact Mish where only requantized int8 values leave the kernel: round((mish(x) [+ add]) * scale) has to be the exact
// form's, the float in between does not.  A short form, x - 2x / (w + 2) as one fused multiply-add behind mish_short's
// reciprocal, is within 8 * 2^-24 |x| of mish_value for every float x: mish_short is within 6 (all 2^32 inputs compared on the
// device, tests/test_gpu_yolo.py), and its last two roundings, of 1 + quotient and of the product, are 1.5 of that.  With t = the
// short form's product with the scale + 128
// both forms round to the same integer wherever t lies further from a rounding boundary k + 1/2 than
// 2^-20 |x scale| + 2^-16, or, with an addend, 2^-20 |x scale| + 2^-21 |t| + 2^-14: twice the bound and the roundings of sum, product
// and t, each at most 2^-24 of what it rounds.  There the conversion to a byte, which rounds and saturates to [0, 255], gives the value of
// quantize_value + 128 whatever its rule for ties.  The few values that lie closer -- about one in ten thousand, and every
// one whose product is large, infinite or NaN -- are evaluated again by the exact chain, a wavefront at a time and only
// where a lane asks; eleven operations and the two transcendental ones a value otherwise.
// word: the 16 values, four int8 to a word.
template <bool WITH_ADD, class Table>
__device__ __forceinline__ void mish_words_for_rounding(const float (&v)[16], const float (&add)[16], float scale, bool half_even,
                                                        uint32_t (&word)[4], const Table &table) {
    typedef float v16f __attribute__((ext_vector_type(16)));
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const float per_x = __builtin_fabsf(__fmul_rn(scale, 0x1p-20f));
    auto product = [&](float x, float a) __attribute__((always_inline)) {
        const float m = __builtin_fmaf(x, mish_minus_quotient(x), x);
        return __builtin_fmaf(WITH_ADD ? __fadd_rn(m, a) : m, scale, 128.f);
    };
    auto is_near = [&](float x, float t) __attribute__((always_inline)) {
        float margin = __builtin_fmaf(__builtin_fabsf(x), per_x, WITH_ADD ? 0x1p-14f : 0x1p-16f);
        if (WITH_ADD) margin = __builtin_fmaf(__builtin_fabsf(t), 0x1p-21f, margin);
        return !(__builtin_fabsf(__fsub_rn(__builtin_amdgcn_fractf(t), 0.5f)) > margin);      // NaN and infinity: near
    };
    unsigned groups = 0;       // words that hold such a value, by wavefront
    static_for<0, 4>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        bool any = false;
        word[g] = 0;
        static_for<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const float t = product(v[4 * g + j], add[4 * g + j]);
            any |= is_near(v[4 * g + j], t);
            word[g] = __builtin_amdgcn_cvt_pk_u8_f32(t, j, word[g]);
        });
        groups |= __builtin_amdgcn_ballot_w64(any) != 0 ? 1u << g : 0u;
    });
    if (groups != 0) {
        v16f x, a;
        v4u w;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = v[r], a[r] = WITH_ADD ? add[r] : 0.f;
#pragma unroll
        for (int g = 0; g < 4; ++g) w[g] = word[g];
#pragma clang loop unroll(disable)
        for (int r = 0; r < 16; ++r) {
            if (!((groups >> (r >> 2)) & 1u)) continue;
            const float xr = x[r], ar = a[r];
            if (is_near(xr, product(xr, ar))) {
                const float m = mish_value(xr, table);
                const int q = quantize_value(__fmul_rn(WITH_ADD ? __fadd_rn(m, ar) : m, scale), half_even);
                const int shift = 8 * (r & 3);
                w[r >> 2] = (w[r >> 2] & ~(255u << shift)) | (unsigned(q + 128) << shift);
            }
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) word[g] = w[g];
    }
    static_for<0, 4>([&](auto gc) { word[decltype(gc)::value] ^= 0x80808080u; });
}

__device__ __forceinline__ float apply_act_conv_i8(float v, int act, float slope, bool in_body) {
    return apply_act(v, act, slope, in_body);
}
// ... for kernel instantiations that layers with the exact Mish are never routed to
__device__ __forceinline__ float apply_act_without_exact_mish(float v, int act, float slope, bool in_body) {
    if (act == TSX_ACT_MISH_FAST) return mish_short_behind_a_branch(v);
    return apply_act_basic(v, act, slope, in_body);
}

#endif  // __HIPCC__

}  // namespace tsx
