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
TSX_MISH_FN double f64_of_bits(uint64_t u) { double d; __builtin_memcpy(&d, &u, 8); return d; }
TSX_MISH_FN uint64_t bits_of_f64(double d) { uint64_t u; __builtin_memcpy(&u, &d, 8); return u; }

// The host's expf: x * 32 / ln2 = k + r, e^x = 2^(k/32) * (1 + r ln2/32 + ...) as a cubic in r, all in double, the
// product rounded to float once (glibc sysdeps/ieee754/flt-32/e_expf.c, the build with fused multiply-adds).  Its
// early returns -- inf, 0, the largest and smallest finite results beyond |x| of 88 -- come out of the same
// arithmetic on the clamped argument: the double result overflows or underflows the float conversion as the host's
// special cases say.  NaN -> NaN.
// exp2_of_32nds: the body of it, from z = x * 32 / ln2, for arguments whose result neither overflows nor needs the clamp.
TSX_MISH_FN float exp2_of_32nds(double z) {
    double kd = z + 0x1.8p+52;                           // the integer nearest to z, in the low mantissa bits
    const uint64_t ki = bits_of_f64(kd);
    kd -= 0x1.8p+52;
    const double r = z - kd;
    const double s = f64_of_bits(exp2f_table[ki & 31] + (ki << 47));
    const double c = __builtin_fma(0x1.c6af84b912394p-5 / 32768.0, r, 0x1.ebfce50fac4f3p-3 / 1024.0);
    const double r2 = r * r;
    double y = __builtin_fma(0x1.62e42ff0c52d6p-1 / 32.0, r, 1.0);
    y = __builtin_fma(c, r2, y);
    return float(y * s);
}
TSX_MISH_FN float expf_host(float x) {
    const double xd = double(__builtin_fminf(__builtin_fmaxf(x, -150.f), 89.f));
    const float e = exp2_of_32nds(0x1.71547652b82fep+5 * xd);
    return x != x ? x : e;
}

// log(s) for a finite double s >= 1, to under 2^-50 relative: s = 2^k m with m in [1, 2), m = (1 + r) / c with the c of m's
// interval, -0.0077 < r <= 2^-6, log s = k ln2 - log c + log(1 + r), the last as r + r^2 p(r) with p the polynomial through
// (log(1 + r) - r) / r^2 at that interval's Chebyshev nodes (2^-52.6 of log(1 + r)).  Rounded to float it is what
// the host's log gives rounded to float: both are far inside half a float ulp of the exact value.
TSX_MISH_FN double log_precise(double s) {
    const uint64_t ix = bits_of_f64(s);
    const uint32_t hi = uint32_t(ix >> 32);
    const int i = int(hi >> 14) & 63;
    const double m = f64_of_bits((uint64_t((hi & 0xfffffu) | 0x3ff00000u) << 32) | uint32_t(ix));
    const double r = __builtin_fma(m, double(log_inverse[i]), -1.0);
    double p = 0x1.1e976e180c123p-3;
    p = __builtin_fma(p, r, -0x1.55535716b7ee6p-3);
    p = __builtin_fma(p, r, 0x1.9999ba4316280p-3);
    p = __builtin_fma(p, r, -0x1.0000000acd4cep-2);
    p = __builtin_fma(p, r, 0x1.55555555413c3p-2);
    p = __builtin_fma(p, r, -0x1.fffffffffffabp-2);
    const double lm = __builtin_fma(r * r, p, r);
    const double kd = double(int(hi >> 20) - 1023);
    // k ln2, ln2 in two parts
    return __builtin_fma(kd, 0x1.62e42fefa38p-1, log_of_interval[i]) + __builtin_fma(kd, 0x1.ef35793c7673p-45, lm);
}

// cpu::Softplus (src/kernels/cpu/softplus.cpp:30-39): float(log(double(expf(x)) + 1.0))
TSX_MISH_FN float softplus_value(float x) {
    const double s = double(expf_host(x)) + 1.0;
    const double l = log_precise(s);
    return s < __builtin_inf() ? float(l) : float(s);   // +inf and NaN pass through
}

// cpu::Tanh (src/kernels/cpu/tanh.cpp:14-23): T(2) * (T(1) / (T(1) + exp(-(T(2) * x)))) - T(1) in float
TSX_MISH_FN float tanh_value(float y) {
    const float u = expf_host(-(2.f * y));
    const float q = div_rn(1.f, 1.f + u);
    return __builtin_fmaf(2.f, q, -1.f);   // 2q is exact: one rounding, fused or not
}

// ---- Mish in one: the composition's values by shorter steps

// log(m) for m in [1, 2) by intervals of 1/256: 4096 times an approximation of 1/m inside the interval, and minus the
// approximation's logarithm.  The first interval has 1 and 0, as in the tables above.
TSX_MISH_TABLE uint16_t mish_inverse_4096ths[256] = {
    4096, 4072, 4056, 4041, 4025, 4010, 3995, 3979, 3964, 3949, 3935, 3920, 3905, 3891, 3876, 3862, 3848, 3834, 3820, 3806, 3792, 3779, 3765, 3752, 3738, 3725, 3712, 3699, 3686, 3673, 3660, 3647,
    3635, 3622, 3610, 3597, 3585, 3573, 3561, 3548, 3537, 3525, 3513, 3501, 3489, 3478, 3466, 3455, 3444, 3432, 3421, 3410, 3399, 3388, 3377, 3366, 3355, 3345, 3334, 3324, 3313, 3303, 3292, 3282,
    3272, 3262, 3251, 3241, 3231, 3221, 3212, 3202, 3192, 3182, 3173, 3163, 3154, 3144, 3135, 3125, 3116, 3107, 3098, 3089, 3080, 3071, 3062, 3053, 3044, 3035, 3026, 3017, 3009, 3000, 2992, 2983,
    2975, 2966, 2958, 2950, 2941, 2933, 2925, 2917, 2909, 2901, 2893, 2885, 2877, 2869, 2861, 2853, 2846, 2838, 2830, 2823, 2815, 2807, 2800, 2792, 2785, 2778, 2770, 2763, 2756, 2749, 2741, 2734,
    2727, 2720, 2713, 2706, 2699, 2692, 2685, 2678, 2672, 2665, 2658, 2651, 2645, 2638, 2631, 2625, 2618, 2612, 2605, 2599, 2592, 2586, 2580, 2573, 2567, 2561, 2554, 2548, 2542, 2536, 2530, 2524,
    2518, 2512, 2506, 2500, 2494, 2488, 2482, 2476, 2470, 2464, 2459, 2453, 2447, 2441, 2436, 2430, 2424, 2419, 2413, 2408, 2402, 2397, 2391, 2386, 2380, 2375, 2370, 2364, 2359, 2354, 2348, 2343,
    2338, 2333, 2328, 2322, 2317, 2312, 2307, 2302, 2297, 2292, 2287, 2282, 2277, 2272, 2267, 2262, 2257, 2253, 2248, 2243, 2238, 2233, 2229, 2224, 2219, 2215, 2210, 2205, 2201, 2196, 2191, 2187,
    2182, 2178, 2173, 2169, 2164, 2160, 2155, 2151, 2147, 2142, 2138, 2133, 2129, 2125, 2120, 2116, 2112, 2108, 2103, 2099, 2095, 2091, 2087, 2083, 2078, 2074, 2070, 2066, 2062, 2058, 2054, 2050,
};
TSX_MISH_TABLE double mish_log_of_interval[256] = {
    0x0.0p+0, 0x1.8121214586b54p-8, 0x1.41929f96832f0p-7, 0x1.bafb16b74919bp-7, 0x1.1e7d80b1fbf41p-6, 0x1.5ba9a5d9ac039p-6,
    0x1.99107b63b81e1p-6, 0x1.dad06ca02682fp-6, 0x1.0c58fa19dfaaap-5, 0x1.2b67c571a29d3p-5, 0x1.487fceb8b26eep-5, 0x1.67c94f2d4bb58p-5,
    0x1.873184bc09592p-5, 0x1.a49da08d3ffa4p-5, 0x1.c441e06f72a9ep-5, 0x1.e1e6713606d07p-5, 0x1.ffa6911ab9301p-5, 0x1.0ec139c5da601p-4,
    0x1.1dbd2643d190bp-4, 0x1.2cc7284fe5f1cp-4, 0x1.3bdf5a7d1ee64p-4, 0x1.49f054cd18720p-4, 0x1.59242ff043d37p-4, 0x1.674f089365a7ap-4,
    0x1.769ef2c6b568dp-4, 0x1.84e40992a480bp-4, 0x1.9335e5d594989p-4, 0x1.a1949e8050083p-4, 0x1.b0004ac1a86acp-4, 0x1.be79020757086p-4,
    0x1.ccfedbfee13a8p-4, 0x1.db91f09680dfep-4, 0x1.e911d663ba274p-4, 0x1.f7be9fedbfde6p-4, 0x1.02ab352ff25f4p-3, 0x1.0a0ea2164af01p-3,
    0x1.10e6a437247b7p-3, 0x1.17c4862a78dfdp-3, 0x1.1ea8520e8e6abp-3, 0x1.2625d1e6ddf57p-3, 0x1.2c81d0a59878fp-3, 0x1.33779819ae5e9p-3,
    0x1.3a73730182ce0p-3, 0x1.41756c0220c82p-3, 0x1.487d8ddca5066p-3, 0x1.4ef51f6466de4p-3, 0x1.56092e02ba516p-3, 0x1.5c8bc079d828ap-3,
    0x1.6313a37335d76p-3, 0x1.6a399dabbd383p-3, 0x1.70ccb9927bcf7p-3, 0x1.77654128f6127p-3, 0x1.7e033d66cd24dp-3, 0x1.84a6b759f512fp-3,
    0x1.8b4fb826ff293p-3, 0x1.91fe49096581bp-3, 0x1.98b27353d7ce7p-3, 0x1.9ecf7d8f3142dp-3, 0x1.a58e729348f43p-3, 0x1.abb55c31693adp-3,
    0x1.b27f3ee67421cp-3, 0x1.b8b027fe249dep-3, 0x1.bf851c067555fp-3, 0x1.c5c0254bf23a6p-3, 0x1.cc000c9db3c52p-3, 0x1.d244d99c85674p-3,
    0x1.d92fd2b1383b6p-3, 0x1.df7f018ce7720p-3, 0x1.e5d32e2e9ce87p-3, 0x1.ec2c60824fbe9p-3, 0x1.f1e75fadf9bdep-3, 0x1.f84a32ead7c35p-3,
    0x1.feb2233ea07cdp-3, 0x1.028f9c7035c1cp-2, 0x1.05761cbf25f1fp-2, 0x1.08b196753a123p-2, 0x1.0b9c8e32d1911p-2, 0x1.0edd060b78081p-2,
    0x1.11cc830ebd9b4p-2, 0x1.1512088e66669p-2, 0x1.180618ef18adfp-2, 0x1.1afc59297024bp-2, 0x1.1df4cc7cf242dp-2, 0x1.20ef7630666d2p-2,
    0x1.23ec5991eba49p-2, 0x1.26eb79f70e869p-2, 0x1.29ecdabcdfa04p-2, 0x1.2cf07f480a155p-2, 0x1.2ff66b04ea9d4p-2, 0x1.32fea167a6d71p-2,
    0x1.360925ec44f5dp-2, 0x1.3915fc16c3c79p-2, 0x1.3bce0507acee9p-2, 0x1.3edf463c1683ep-2, 0x1.419b423d5e8c7p-2, 0x1.44b0fb5af4f43p-2,
    0x1.4770f5f6b9fa6p-2, 0x1.4a8b341552b09p-2, 0x1.4d4f3908901a0p-2, 0x1.501528da1f968p-2, 0x1.533624b59ca35p-2, 0x1.560030809c75ap-2,
    0x1.58cc2f91489f5p-2, 0x1.5b9a24a3bd662p-2, 0x1.5e6a1279dbb70p-2, 0x1.613bfbdb596a0p-2, 0x1.640fe395d1c02p-2, 0x1.66e5cc7cd61b4p-2,
    0x1.69bdb969fef18p-2, 0x1.6c97ad3cfcfd9p-2, 0x1.6f73aadbaaab9p-2, 0x1.7251b5321dc53p-2, 0x1.74d5aefd66d5cp-2, 0x1.77b79922bd37ep-2,
    0x1.7a9b9889f19e2p-2, 0x1.7d24cfd3b931cp-2, 0x1.800cbf3ed1cc3p-2, 0x1.82f6ccabaeb52p-2, 0x1.85855776dcbfbp-2, 0x1.8873658327ccfp-2,
    0x1.8b0575aab1fc4p-2, 0x1.8d992dc8824e5p-2, 0x1.908d2ea7d9512p-2, 0x1.93247a7c99b53p-2, 0x1.95bd750ee3ed3p-2, 0x1.9858208f94f57p-2,
    0x1.9b541e1687a3fp-2, 0x1.9df270c1914a8p-2, 0x1.a0927b59da6e2p-2, 0x1.a33440224fa79p-2, 0x1.a5d7c16257437p-2, 0x1.a87d0165dd199p-2,
    0x1.ab24027d5e8b0p-2, 0x1.adccc6fdf6a81p-2, 0x1.b07751416a7f4p-2, 0x1.b323a3a635948p-2, 0x1.b56fa04462909p-2, 0x1.b81f481bd74aap-2,
    0x1.bad0bef3db165p-2, 0x1.bd84073d8ec2bp-2, 0x1.bfd602aa3fa9fp-2, 0x1.c28cb1e4d32fdp-2, 0x1.c54539a6abcd2p-2, 0x1.c79bba4d55a7cp-2,
    0x1.ca57b64e9db05p-2, 0x1.ccb130a5cebb0p-2, 0x1.cf70a9b6d380fp-2, 0x1.d1cd255af9931p-2, 0x1.d490246defa6bp-2, 0x1.d6efa918d25cdp-2,
    0x1.d9509707ae52fp-2, 0x1.dc18cccbdcb84p-2, 0x1.de7ccf4216d6ep-2, 0x1.e0e2405a6cfd5p-2, 0x1.e3afc0a49ff40p-2, 0x1.e6185206d516ep-2,
    0x1.e882578823d52p-2, 0x1.eaedd2eac990cp-2, 0x1.ed5ac5f436be3p-2, 0x1.efc9326d16ab9p-2, 0x1.f2391a2157600p-2, 0x1.f4aa7ee03192dp-2,
    0x1.f71d627c30bb0p-2, 0x1.f991c6cb3b379p-2, 0x1.fc07ada69a910p-2, 0x1.fe7f18eb03d3ep-2, 0x1.007c053c5002ep-1, 0x1.01b942198a5a1p-1,
    0x1.02f74400c64ebp-1, 0x1.04360be7603adp-1, 0x1.05404a6ea6442p-1, 0x1.06807fd750858p-1, 0x1.07c17e0056e7cp-1, 0x1.090345e60f709p-1,
    0x1.0a10074cf9019p-1, 0x1.0b5343a234477p-1, 0x1.0c974c89431cep-1, 0x1.0da5f0f46ba3ap-1, 0x1.0eeb738a67874p-1, 0x1.0ffb54213a476p-1,
    0x1.114253da97d9fp-1, 0x1.125373832f061p-1, 0x1.139bf3e094003p-1, 0x1.14ae558b4a92dp-1, 0x1.15f85a19c765bp-1, 0x1.170c00c169b50p-1,
    0x1.18203c20dd133p-1, 0x1.196c7bc4b1f3bp-1, 0x1.1a820089a2156p-1, 0x1.1b981c0c9653dp-1, 0x1.1ce69e8bb106bp-1, 0x1.1dfe07f3d1dabp-1,
    0x1.1f160a2ad0da4p-1, 0x1.202ea5d82d3d7p-1, 0x1.2147dba47a394p-1, 0x1.229a1bc5ebac3p-1, 0x1.23b4a6f9d8688p-1, 0x1.24cfce6f80d9ap-1,
    0x1.25eb92d41992dp-1, 0x1.2707f4d5f7c41p-1, 0x1.2824f52493bd3p-1, 0x1.294294708b773p-1, 0x1.2a60d36ba5253p-1, 0x1.2b7fb2c8d1cc1p-1,
    0x1.2c9f333c2fe1dp-1, 0x1.2dbf557b0df43p-1, 0x1.2ee01a3bed567p-1, 0x1.3001823684d73p-1, 0x1.31238e23c37dbp-1, 0x1.320c0e364a4a6p-1,
    0x1.332f4314ad796p-1, 0x1.34531df21cfe4p-1, 0x1.35779f8c43d6ep-1, 0x1.369cc8a212cdep-1, 0x1.3787c8fe53181p-1, 0x1.38ae2171976e7p-1,
    0x1.39d5237e045a5p-1, 0x1.3ac19fc17fe50p-1, 0x1.3be9d503533b5p-1, 0x1.3d12b60622748p-1, 0x1.3e00b304f5387p-1, 0x1.3f2acb27ed6c7p-1,
    0x1.4055913e4b42dp-1, 0x1.414513e448ca2p-1, 0x1.42711518df545p-1, 0x1.436194e12b6bfp-1, 0x1.448ed3cf71355p-1, 0x1.458052d35471ap-1,
    0x1.46aed21f117fcp-1, 0x1.47a1527e8a2d3p-1, 0x1.48d114d3fb884p-1, 0x1.49c498b5da63fp-1, 0x1.4ab890a0bcfa7p-1, 0x1.4bea2a5bdbe87p-1,
    0x1.4cdf28f10ac46p-1, 0x1.4e120c62f195fp-1, 0x1.4f0813da673dcp-1, 0x1.4ffe91c3f6a1bp-1, 0x1.513356667fc57p-1, 0x1.522ae0738a3d8p-1,
    0x1.5322e26867857p-1, 0x1.541b5cb979809p-1, 0x1.55529f92da1c1p-1, 0x1.564c2a6059fe8p-1, 0x1.57462f08e7df5p-1, 0x1.5840ae03c0203p-1,
    0x1.593ba7c8ce7adp-1, 0x1.5a371cd0af593p-1, 0x1.5b721d295f10fp-1, 0x1.5c6ea94431ef9p-1, 0x1.5d6bb22ea86f6p-1, 0x1.5e6938645d390p-1,
    0x1.5f673c61a2ed2p-1, 0x1.6065bea385926p-1, 0x1.6164bfa7cc06bp-1, 0x1.62643fecf9743p-1,
};

// where mish_value finds 2^(i/32), two over the interval's inverse approximation and its logarithm: in memory, or a copy
struct MishTablesInMemory {
    TSX_MISH_MEMBER uint64_t exp2(uint32_t i) const { return exp2f_table[i]; }
    TSX_MISH_MEMBER double twice_inverse(int i) const { return double(mish_inverse_4096ths[i]) * (1.0 / 2048); }
    TSX_MISH_MEMBER double log_of(int i) const { return mish_log_of_interval[i]; }
};

// The addends of the first steps of its two polynomials: a caller that evaluates many keeps them in vector registers, since an
// instruction reads one pair of scalar registers only.
struct MishAddends {
    double exp2 = 0x1.ebfce50fac4f3p-3 / 1024.0, log = -0x1.0000276b2de2cp-2;
};

#ifdef __HIP_DEVICE_COMPILE__
// 1 / d rounded to nearest for d in [1, 2]: no scaling is needed there, one Newton step on the device's reciprocal.  (Every d that
// occurs gives the division's bits in Mish: the comparison of mish_value with the operators, which divide, for all 2^32 floats.)
TSX_MISH_FN float reciprocal_rn_1_2(float d) {
    const float a = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, a, 1.f), a, a);
}
// s = half_mantissa * 2^(exponent), half_mantissa in [1/2, 1)
TSX_MISH_FN double half_mantissa(double s) { return __builtin_amdgcn_frexp_mant(s); }
TSX_MISH_FN int half_exponent(double s) { return __builtin_amdgcn_frexp_exp(s); }
TSX_MISH_FN float clamped(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }
// hi + (k << 15) as an instruction: as an addition to the high half of 64 bits the compiler makes it one of all 64, and moves
TSX_MISH_FN uint32_t add_exponent(uint32_t hi, uint32_t k) {
    asm("v_lshl_add_u32 %0, %1, 15, %0" : "+v"(hi) : "v"(k));
    return hi;
}
#else
TSX_MISH_FN float reciprocal_rn_1_2(float d) { return 1.f / d; }
TSX_MISH_FN double half_mantissa(double s) { return f64_of_bits((bits_of_f64(s) & 0xfffffffffffffULL) | 0x3fe0000000000000ULL); }
TSX_MISH_FN int half_exponent(double s) { return int(bits_of_f64(s) >> 52) - 1022; }
TSX_MISH_FN float clamped(float x, float lo, float hi) { return __builtin_fminf(__builtin_fmaxf(x, lo), hi); }
TSX_MISH_FN uint32_t add_exponent(uint32_t hi, uint32_t k) { return hi + (k << 15); }
#endif

// exp2_of_32nds with its polynomial in another order: 2^(k/32) + 2^(k/32) r (C2 + r (C1 + r C0))
template <class Table>
TSX_MISH_FN float mish_exp2(double z, const Table &table, const MishAddends &add) {
    double kd = z + 0x1.8p+52;
    const uint32_t ki = uint32_t(bits_of_f64(kd));
    kd -= 0x1.8p+52;
    const double r = z - kd;
    uint32_t half[2];
    const uint64_t t = table.exp2(ki & 31);
    __builtin_memcpy(half, &t, 8);
    half[1] = add_exponent(half[1], ki);
    double s;
    __builtin_memcpy(&s, half, 8);
    double p = __builtin_fma(0x1.c6af84b912394p-5 / 32768.0, r, add.exp2);
    p = __builtin_fma(p, r, 0x1.62e42ff0c52d6p-1 / 32.0);
    return float(__builtin_fma(s * r, p, s));
}

// log(s) for a finite double s >= 1, to 2^-46 relative: s = 2^k m, m = (1 + r) / c, |r| <= 2^-8, log s = k ln2 - log c + r (1 + r p(r))
// with p through (log(1 + r) - r) / r^2 at the Chebyshev nodes of all r that occur.
template <class Table>
TSX_MISH_FN double mish_log(double s, const Table &table, const MishAddends &add) {
    const int i = int(uint32_t(bits_of_f64(s) >> 32) >> 12) & 255;
    const double r = __builtin_fma(half_mantissa(s), table.twice_inverse(i), -1.0);
    double p = __builtin_fma(0x1.9852ea3ae0af9p-3, r, add.log);
    p = __builtin_fma(p, r, 0x1.5555557b13110p-2);
    p = __builtin_fma(p, r, -0x1.fffffffffe03ep-2);
    return __builtin_fma(r, __builtin_fma(r, p, 1.0), __builtin_fma(double(half_exponent(s) - 1), 0x1.62e42fefa39efp-1, table.log_of(i)));
}

// x * tanh_value(softplus_value(x)), bit for bit (a NaN aside, of which the result is one too) for all 2^32 floats:
// tests/test_gpu_yolo.py compares them on the device.  What the composition needs only at the ends of the float range is left out: below -18.1
// the tangent is 0 and above 10 it is 1, so the argument is clamped to these once (a NaN too: the product with x makes it one
// again); the exponentials then neither overflow nor vanish, e^x + 1 is finite, and the divisor 1 + e^(-2y) lies in [1, 2].  -2y *
// 32 / ln2 is the host's product, scaled by a power of two.  The exponentials have to round as the host's do, and the logarithm,
// which rounds to a float, to be far closer than a float: 2^-46 is enough for every float that occurs.  50 instructions and three table reads;
// 62 with the logarithm from 64 intervals to 2^-50, two Newton steps and 64-bit additions of exponents (values in
// registers, all CUs: 230 -> 185 cycles a wavefront's 64 values).
template <class Table = MishTablesInMemory>
TSX_MISH_FN float mish_value(float x, const Table &table = Table(), const MishAddends &add = MishAddends()) {
    const double xd = double(clamped(x, -18.1f, 10.f));
    const float e = mish_exp2(0x1.71547652b82fep+5 * xd, table, add);
    const float y = float(mish_log(double(e) + 1.0, table, add));
    const float u = mish_exp2(-0x1.71547652b82fep+6 * double(y), table, add);
    return x * __builtin_fmaf(2.f, reciprocal_rn_1_2(1.f + u), -1.f);
}

}  // namespace tsx
