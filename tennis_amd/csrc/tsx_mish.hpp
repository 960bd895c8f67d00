// Mish as TenniS graphs compose it -- mul(x, tanh(softplus(x))) -- in the host's arithmetic:
//   softplus(x) = float(log(double(expf(x)) + 1.0))          src/kernels/cpu/softplus.cpp:30-39
//   tanh(y)     = 2 * (1 / (1 + expf(-(2 y)))) - 1 in float  src/kernels/cpu/tanh.cpp:14-23
// The host's expf and log are its C library's (glibc 2.35 on the reference's x86-64 build).  Here expf is restated
// operation for operation and log is evaluated far beyond float precision, so every rounded intermediate of the
// chain, and with it the result, is the host's bit for bit.
//
// This header compiles for the device (hipcc) and, unchanged, for the host (g++ -ffp-contract=off): the host build
// exists so that a dense sweep over the floats can hold these very functions against the C library's chain without
// a GPU.  Everything is written with explicit fused multiply-adds and otherwise plain IEEE operations; the build
// must not contract or reassociate (-ffp-contract=off, no fast-math).
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define TSX_MISH_FN __device__ __forceinline__
#define TSX_MISH_MEMBER __device__ __forceinline__
#define TSX_MISH_TABLE static __device__ const
#else
#define TSX_MISH_FN static inline
#define TSX_MISH_MEMBER inline
#define TSX_MISH_TABLE static const
#endif

namespace tsx {

// 2^(i/32) as doubles, less i << 47 (the table of glibc's expf, sysdeps/ieee754/flt-32/e_exp2f_data.c)
TSX_MISH_TABLE uint64_t exp2f_table[32] = {
    0x3ff0000000000000ULL, 0x3fefd9b0d3158574ULL, 0x3fefb5586cf9890fULL, 0x3fef9301d0125b51ULL,
    0x3fef72b83c7d517bULL, 0x3fef54873168b9aaULL, 0x3fef387a6e756238ULL, 0x3fef1e9df51fdee1ULL,
    0x3fef06fe0a31b715ULL, 0x3feef1a7373aa9cbULL, 0x3feedea64c123422ULL, 0x3feece086061892dULL,
    0x3feebfdad5362a27ULL, 0x3feeb42b569d4f82ULL, 0x3feeab07dd485429ULL, 0x3feea47eb03a5585ULL,
    0x3feea09e667f3bcdULL, 0x3fee9f75e8ec5f74ULL, 0x3feea11473eb0187ULL, 0x3feea589994cce13ULL,
    0x3feeace5422aa0dbULL, 0x3feeb737b0cdc5e5ULL, 0x3feec49182a3f090ULL, 0x3feed503b23e255dULL,
    0x3feee89f995ad3adULL, 0x3feeff76f2fb5e47ULL, 0x3fef199bdd85529cULL, 0x3fef3720dcef9069ULL,
    0x3fef5818dcfba487ULL, 0x3fef7c97337b9b5fULL, 0x3fefa4afa2a490daULL, 0x3fefd0765b6e4540ULL,
};

// log(m) for m in [1, 2) by intervals of 1/64: an approximation of 1/m inside the interval that a float holds exactly, and
// minus its logarithm.  The first interval has 1 and 0, so that log(1 + f) keeps its relative accuracy for small f.
TSX_MISH_TABLE float log_inverse[64] = {
    4096.f / 4096, 4002.f / 4096, 3942.f / 4096, 3884.f / 4096, 3827.f / 4096, 3772.f / 4096, 3718.f / 4096, 3666.f / 4096,
    3616.f / 4096, 3567.f / 4096, 3519.f / 4096, 3472.f / 4096, 3427.f / 4096, 3383.f / 4096, 3339.f / 4096, 3297.f / 4096,
    3256.f / 4096, 3216.f / 4096, 3178.f / 4096, 3139.f / 4096, 3102.f / 4096, 3066.f / 4096, 3031.f / 4096, 2996.f / 4096,
    2962.f / 4096, 2929.f / 4096, 2897.f / 4096, 2865.f / 4096, 2834.f / 4096, 2804.f / 4096, 2774.f / 4096, 2745.f / 4096,
    2717.f / 4096, 2689.f / 4096, 2661.f / 4096, 2635.f / 4096, 2608.f / 4096, 2583.f / 4096, 2558.f / 4096, 2533.f / 4096,
    2509.f / 4096, 2485.f / 4096, 2461.f / 4096, 2439.f / 4096, 2416.f / 4096, 2394.f / 4096, 2372.f / 4096, 2351.f / 4096,
    2330.f / 4096, 2310.f / 4096, 2289.f / 4096, 2270.f / 4096, 2250.f / 4096, 2231.f / 4096, 2212.f / 4096, 2194.f / 4096,
    2175.f / 4096, 2158.f / 4096, 2140.f / 4096, 2123.f / 4096, 2106.f / 4096, 2089.f / 4096, 2072.f / 4096, 2056.f / 4096,
};
TSX_MISH_TABLE double log_of_interval[64] = {
    0x0.0p+0, 0x1.7c61b1cf5dee0p-6, 0x1.39f07ba0ebd62p-5, 0x1.b35dd9b58baadp-5,
    0x1.163d6ef957a03p-4, 0x1.518874226130ap-4, 0x1.8c985e9b9ec84p-4, 0x1.c6494a2e418a6p-4,
    0x1.fe89139dbd566p-4, 0x1.1b35ae3b81dbfp-3, 0x1.36f4c27577593p-3, 0x1.527e5e4a1b58dp-3,
    0x1.6d35fee52b83bp-3, 0x1.87ad07c493478p-3, 0x1.a27cc30640ecbp-3, 0x1.bc69684aee63ep-3,
    0x1.d60a17f903515p-3, 0x1.ef5ade4dcffe6p-3, 0x1.03d95a1d67686p-2, 0x1.107e404ab0f81p-2,
    0x1.1ca28c64bae54p-2, 0x1.2896a13e086a4p-2, 0x1.34585a594b8adp-2, 0x1.403d086cea79cp-2,
    0x1.4becf95d97913p-2, 0x1.5765f1749da6bp-2, 0x1.62a5afc06121fp-2, 0x1.6e056aa4421d5p-2,
    0x1.792955fdf47a2p-2, 0x1.840f1e12667f0p-2, 0x1.8f12e873862c8p-2, 0x1.99d5d8130607dp-2,
    0x1.a4558a1c9b824p-2, 0x1.aef113b0bc778p-2, 0x1.b9a90a06bcb3ep-2, 0x1.c3b6fb361e301p-2,
    0x1.ce42f18064743p-2, 0x1.d81ff2cce8a4ep-2, 0x1.e21582ecdbf74p-2, 0x1.ec241d5e2ffd0p-2,
    0x1.f5e3c0b5425c6p-2, 0x1.ffbb60ca863b3p-2, 0x1.04d5ba679ac9bp-1, 0x1.096eb58872addp-1,
    0x1.0e4898611cce1p-1, 0x1.12f799594efbcp-1, 0x1.17b1ac17cbd5bp-1, 0x1.1c3f41fa97c6bp-1,
    0x1.20d74d2fbafe5p-1, 0x1.25413d529caeep-1, 0x1.29ee409f15440p-1, 0x1.2e32c3d74d58bp-1,
    0x1.32bab3a7b21e8p-1, 0x1.37123b54987b6p-1, 0x1.3b7344be40311p-1, 0x1.3fa238ac248a5p-1,
    0x1.44163ef7283d9p-1, 0x1.481abdce327f6p-1, 0x1.4c649aff0ee16p-1, 0x1.5079fd47366f8p-1,
    0x1.5497c729233afp-1, 0x1.58be1b857aebep-1, 0x1.5ced1e17c35c5p-1, 0x1.60e52f45788e3p-1,
};

#ifdef __HIPCC__
TSX_MISH_FN float div_rn(float a, float b) { return __fdiv_rn(a, b); }   // IEEE division whatever the build's default
#else
TSX_MISH_FN float div_rn(float a, float b) { return a / b; }
#endif
// where expf_host finds 2^(i/32), and log_precise its interval: these tables in memory, or whatever holds a copy of them (on
// the device, the workgroup's LDS)
struct MishTablesInMemory {
    TSX_MISH_MEMBER uint64_t exp2(uint32_t i) const { return exp2f_table[i]; }
    TSX_MISH_MEMBER double inverse(int i) const { return double(log_inverse[i]); }
    TSX_MISH_MEMBER double log_of(int i) const { return log_of_interval[i]; }
};

TSX_MISH_FN double f64_of_bits(uint64_t u) { double d; __builtin_memcpy(&d, &u, 8); return d; }
TSX_MISH_FN uint64_t bits_of_f64(double d) { uint64_t u; __builtin_memcpy(&u, &d, 8); return u; }

// The host's expf: x * 32 / ln2 = k + r, e^x = 2^(k/32) * (1 + r ln2/32 + ...) as a cubic in r, all in double, the
// product rounded to float once (glibc sysdeps/ieee754/flt-32/e_expf.c, the build with fused multiply-adds).  Its
// early returns -- inf, 0, the largest and smallest finite results beyond |x| of 88 -- come out of the same
// arithmetic on the clamped argument: the double result overflows or underflows the float conversion as the host's
// special cases say.  NaN -> NaN.
// exp2_of_32nds: the body of it, from z = x * 32 / ln2, for arguments whose result neither overflows nor needs the clamp.
template <class Table = MishTablesInMemory>
TSX_MISH_FN float exp2_of_32nds(double z, const Table &table = Table()) {
    double kd = z + 0x1.8p+52;                           // the integer nearest to z, in the low mantissa bits
    const uint64_t ki = bits_of_f64(kd);
    kd -= 0x1.8p+52;
    const double r = z - kd;
    const double s = f64_of_bits(table.exp2(uint32_t(ki) & 31) + (ki << 47));
    const double c = __builtin_fma(0x1.c6af84b912394p-5 / 32768.0, r, 0x1.ebfce50fac4f3p-3 / 1024.0);
    const double r2 = r * r;
    double y = __builtin_fma(0x1.62e42ff0c52d6p-1 / 32.0, r, 1.0);
    y = __builtin_fma(c, r2, y);
    return float(y * s);
}
template <class Table = MishTablesInMemory>
TSX_MISH_FN float expf_host(float x, const Table &table = Table()) {
    const double xd = double(__builtin_fminf(__builtin_fmaxf(x, -150.f), 89.f));
    const float e = exp2_of_32nds(0x1.71547652b82fep+5 * xd, table);
    return x != x ? x : e;
}

// log(s) for a finite double s >= 1, to under 2^-50 relative: s = 2^k m with m in [1, 2), m = (1 + r) / c with the c of m's
// interval, -0.0077 < r <= 2^-6, log s = k ln2 - log c + log(1 + r), the last as r + r^2 p(r) with p the polynomial through
// (log(1 + r) - r) / r^2 at that interval's Chebyshev nodes (2^-52.6 of log(1 + r)).  Rounded to float it is what
// the host's log gives rounded to float: both are far inside half a float ulp of the exact value.
template <class Table = MishTablesInMemory>
TSX_MISH_FN double log_precise(double s, const Table &table = Table()) {
    const uint64_t ix = bits_of_f64(s);
    const uint32_t hi = uint32_t(ix >> 32);
    const int i = int(hi >> 14) & 63;
    const double m = f64_of_bits((uint64_t((hi & 0xfffffu) | 0x3ff00000u) << 32) | uint32_t(ix));
    const double r = __builtin_fma(m, table.inverse(i), -1.0);
    double p = 0x1.1e976e180c123p-3;
    p = __builtin_fma(p, r, -0x1.55535716b7ee6p-3);
    p = __builtin_fma(p, r, 0x1.9999ba4316280p-3);
    p = __builtin_fma(p, r, -0x1.0000000acd4cep-2);
    p = __builtin_fma(p, r, 0x1.55555555413c3p-2);
    p = __builtin_fma(p, r, -0x1.fffffffffffabp-2);
    const double lm = __builtin_fma(r * r, p, r);
    const double kd = double(int(hi >> 20) - 1023);
    // k ln2, ln2 in two parts
    return __builtin_fma(kd, 0x1.62e42fefa38p-1, table.log_of(i)) + __builtin_fma(kd, 0x1.ef35793c7673p-45, lm);
}

// cpu::Softplus (src/kernels/cpu/softplus.cpp:30-39): float(log(double(expf(x)) + 1.0))
template <class Table = MishTablesInMemory>
TSX_MISH_FN float softplus_value(float x, const Table &table = Table()) {
    const double s = double(expf_host(x, table)) + 1.0;
    const double l = log_precise(s, table);
    return s < __builtin_inf() ? float(l) : float(s);   // +inf and NaN pass through
}

// cpu::Tanh (src/kernels/cpu/tanh.cpp:14-23): T(2) * (T(1) / (T(1) + exp(-(T(2) * x)))) - T(1) in float
template <class Table = MishTablesInMemory>
TSX_MISH_FN float tanh_value(float y, const Table &table = Table()) {
    const float u = expf_host(-(2.f * y), table);
    const float q = div_rn(1.f, 1.f + u);
    return __builtin_fmaf(2.f, q, -1.f);   // 2q is exact: one rounding, fused or not
}

// 1 / d rounded to nearest for d in [1, 2]: no scaling is needed there, two Newton steps on the device's reciprocal.  (Every d that
// occurs gives the division's bits in Mish: tests/test_gpu_yolo.py, which holds mish_value against x tanh(softplus(x)) by
// the functions above for all floats on the device.)
#ifdef __HIP_DEVICE_COMPILE__
TSX_MISH_FN float reciprocal_rn_1_2(float d) {
    const float a = __builtin_amdgcn_rcpf(d);
    const float b = __builtin_fmaf(__builtin_fmaf(-d, a, 1.f), a, a);
    return __builtin_fmaf(__builtin_fmaf(-d, b, 1.f), b, b);
}
#else
TSX_MISH_FN float reciprocal_rn_1_2(float d) { return 1.f / d; }
#endif

// x * tanh_value(softplus_value(x)), the same bits without what the composition needs only at the ends of the float range:
// below -20 the tangent is 0 and above 40 it is 1 whatever the argument, so the argument is clamped to these once (a NaN
// too: the product with x makes it one again); the exponentials then neither overflow nor vanish, e^x + 1 is finite, and
// the divisor 1 + e^(-2y) lies in [1, 2].  -2y * 32 / ln2 is the host's product, scaled by a power of two.  56 double- and
// single-precision operations and four table reads, where the composition has 92 and (with tables in the lanes) seven.
template <class Table = MishTablesInMemory>
TSX_MISH_FN float mish_value(float x, const Table &table = Table()) {
    const double xd = double(__builtin_fminf(__builtin_fmaxf(x, -20.f), 40.f));
    const float e = exp2_of_32nds(0x1.71547652b82fep+5 * xd, table);
    const float y = float(log_precise(double(e) + 1.0, table));
    const float u = exp2_of_32nds(-0x1.71547652b82fep+6 * double(y), table);
    return x * __builtin_fmaf(2.f, reciprocal_rn_1_2(1.f + u), -1.f);
}

}  // namespace tsx
