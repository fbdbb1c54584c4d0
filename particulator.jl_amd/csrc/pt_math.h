// pt_math.h -- the step's square roots, divisions, logarithm and sine/cosine in FP64.
//
// The step kernel is bound by instruction issue (every FP64 operation, and every scalar one
// of a wave that is alone on its SIMD, takes an issue slot of four cycles), so these are
// written for few instructions:
//   * sqrt and division: the correctly rounded Newton/Goldschmidt sequences without the
//     scaling that only operands near the ends of the exponent range need (the results are
//     the same for 2^-767 < x < 2^1000, and for exponents of quotient and divisor within
//     +-1000, far beyond the step's values; zero, infinity and NaN are passed on as IEEE
//     has them where the callers can meet them): 15 instead of 22 and 9 instead of 12
//     instructions, and a shared reciprocal (`Recip`) costs 3 per further quotient;
//   * log: table-driven (P. T. P. Tang, ACM TOMS 16 (1990) 378-400) with 128 intervals, about
//     30 instead of 98 instructions, error 0.54 instead of 0.64 ulp;
//   * sine and cosine of an azimuth in [0, 2 pi]: Cody-Waite reduction in two parts and
//     minimax polynomials, about 50 instead of 155 instructions, error 0.75 instead of
//     0.78 ulp (all errors: the largest over 2.5 x 10^7 arguments).
// The same source compiles for the host, where the hardware's approximations of 1/x and
// 1/sqrt(x) are replaced by ones of the same quality, so that a CPU test can compare the
// sequences with IEEE arithmetic and with higher precision.
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define PT_HD __host__ __device__ __forceinline__
#else
#define PT_HD inline
#endif

namespace pt {

#if defined(__HIP_DEVICE_COMPILE__)
PT_HD double approx_rcp(double x) { return __builtin_amdgcn_rcp(x); }
PT_HD double approx_rsq(double x) { return __builtin_amdgcn_rsq(x); }
PT_HD double div_fixup(double q, double b, double a) { return __builtin_amdgcn_div_fixup(q, b, a); }
PT_HD double frexp_mant(double x) { return __builtin_amdgcn_frexp_mant(x); }
PT_HD int frexp_exp(double x) { return __builtin_amdgcn_frexp_exp(x); }
PT_HD bool zero_or_inf(double x) { return __builtin_amdgcn_class(x, 0x60 | 0x200); }  // +-0, +inf
PT_HD double round_even(double x) { return __builtin_rint(x); }
PT_HD double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }
PT_HD uint32_t high_word(double x) { return (uint32_t)__double2hiint(x); }
PT_HD double flip_sign(double x, uint32_t signbit) {
    return __hiloint2double(__double2hiint(x) ^ (int)signbit, __double2loint(x));
}
#else
PT_HD double approx_rcp(double x) { return (1.0 / x) * (1.0 + 0x1p-27); }
PT_HD double approx_rsq(double x) { return (1.0 / sqrt(x)) * (1.0 - 0x1p-27); }
PT_HD double div_fixup(double q, double b, double a) {
    return (b == 0.0 || isinf(b) || isinf(a) || isnan(a) || isnan(b) || a == 0.0) ? a / b : q;
}
PT_HD double frexp_mant(double x) {
    int e;
    return frexp(x, &e);
}
PT_HD int frexp_exp(double x) {
    int e = 0;
    if (x == x && !isinf(x)) (void)frexp(x, &e);
    return e;
}
PT_HD bool zero_or_inf(double x) { return x == 0.0 || (isinf(x) && x > 0); }
PT_HD double round_even(double x) { return nearbyint(x); }
PT_HD double fused(double a, double b, double c) { return fma(a, b, c); }
PT_HD uint32_t high_word(double x) {
    uint64_t b;
    memcpy(&b, &x, 8);
    return (uint32_t)(b >> 32);
}
PT_HD double flip_sign(double x, uint32_t signbit) {
    uint64_t b;
    memcpy(&b, &x, 8);
    b ^= (uint64_t)signbit << 32;
    memcpy(&x, &b, 8);
    return x;
}
#endif

// sqrt(x): one step of Goldschmidt's iteration from the hardware's 1/sqrt(x), then two
// corrections of the root by its exact remainder (P. Markstein, "Software division and square
// root using Goldschmidt's algorithms", Proc. 6th Conf. on Real Numbers and Computers (2004)
// 146-157)
PT_HD double qsqrt(double x) {
    const double y = approx_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fused(-h, g, 0.5);
    g = fused(g, e, g);
    h = fused(h, e, h);
    g = fused(fused(-g, g, x), h, g);
    g = fused(fused(-g, g, x), h, g);
    return zero_or_inf(x) ? x : g;
}

// 1/b to within an ulp, and quotients by it: each is corrected by its exact remainder, which
// rounds it correctly (Markstein, IBM J. Res. Dev. 34 (1990) 111-119)
struct Recip {
    double b, r;
    PT_HD explicit Recip(double d) : b(d) {
        double y = approx_rcp(d);
        y = fused(fused(-d, y, 1.0), y, y);
        r = fused(fused(-d, y, 1.0), y, y);
    }
    // a / b for finite a and finite, nonzero b
    PT_HD double operator()(double a) const {
        const double q = a * r;
        return fused(fused(-b, q, a), r, q);
    }
    PT_HD double inverse() const { return fused(fused(-b, r, 1.0), r, r); }
};
PT_HD double qdiv(double a, double b) { return Recip(b)(a); }
// a / b with zero, infinite and NaN operands as IEEE has them
PT_HD double qdiv_any(double a, double b) { return div_fixup(Recip(b)(a), b, a); }

// log(x) for positive normal x.  x = 2^k m with m in [3/4, 3/2); the interval of m gives c ~
// 1/m and -log(c) in two parts, r = m c - 1 is small (below 2^-7; c has 8 bits after the
// point, so that r is exact), and log(x) = k log 2 -
// log(c) + r + r^2 p(r).  The intervals beside 1 have c = 1, so that log keeps its relative
// accuracy there.  `c` holds the factor 2 of the intervals below 3/4 (frexp gives m in
// [1/2, 1)).
//
// The coefficients of log and of sine and cosine stand in the same table: as literals each
// would take two more instructions (a 64-bit literal is no operand), from LDS two come with
// one read.
constexpr int LOG_N = 128;
constexpr int MATH_LO = 2 * LOG_N;        // {c, high part} pairs, then the low parts
constexpr int MATH_LOG = 3 * LOG_N;       // log 2 in two parts, then p from its highest term
constexpr int MATH_SIN = MATH_LOG + 8;    // 2/pi, pi/2 in three parts, then sine and cosine
constexpr int MATH_DOUBLES = MATH_SIN + 18;
#define PT_MATH_TABLE \
    0x1.0000000000000p+1, 0x0.0p+0, \
    0x1.fa00000000000p+0, 0x1.82448a3880000p-7, \
    0x1.f600000000000p+0, 0x1.432a925980000p-6, \
    0x1.f200000000000p+0, 0x1.c63d2ec150000p-6, \
    0x1.ee00000000000p+0, 0x1.252f32f8d0000p-5, \
    0x1.ea00000000000p+0, 0x1.67c94f2d48000p-5, \
    0x1.e800000000000p+0, 0x1.894aa149f8000p-5, \
    0x1.e400000000000p+0, 0x1.ccb73cddd8000p-5, \
    0x1.e000000000000p+0, 0x1.08598b59e4000p-4, \
    0x1.dc00000000000p+0, 0x1.2aa04a4470000p-4, \
    0x1.da00000000000p+0, 0x1.3bdf5a7d20000p-4, \
    0x1.d600000000000p+0, 0x1.5e95a4d978000p-4, \
    0x1.d200000000000p+0, 0x1.8197e2f410000p-4, \
    0x1.d000000000000p+0, 0x1.9335e5d594000p-4, \
    0x1.cc00000000000p+0, 0x1.b6ac88dad4000p-4, \
    0x1.c800000000000p+0, 0x1.da72763844000p-4, \
    0x1.c600000000000p+0, 0x1.ec739830a0000p-4, \
    0x1.c200000000000p+0, 0x1.08598b59e4000p-3, \
    0x1.c000000000000p+0, 0x1.1178e8227e000p-3, \
    0x1.bc00000000000p+0, 0x1.23d712a49c000p-3, \
    0x1.ba00000000000p+0, 0x1.2d1610c868000p-3, \
    0x1.b600000000000p+0, 0x1.3fb45a5992000p-3, \
    0x1.b400000000000p+0, 0x1.4913d8333c000p-3, \
    0x1.b000000000000p+0, 0x1.5bf406b544000p-3, \
    0x1.ae00000000000p+0, 0x1.6574ebe8c2000p-3, \
    0x1.aa00000000000p+0, 0x1.7898d85444000p-3, \
    0x1.a800000000000p+0, 0x1.823c16551a000p-3, \
    0x1.a600000000000p+0, 0x1.8beafeb390000p-3, \
    0x1.a200000000000p+0, 0x1.9f6c40708a000p-3, \
    0x1.a000000000000p+0, 0x1.a93ed3c8ae000p-3, \
    0x1.9e00000000000p+0, 0x1.b31d8575bc000p-3, \
    0x1.9a00000000000p+0, 0x1.c6ffbc6f00000p-3, \
    0x1.9800000000000p+0, 0x1.d1037f2656000p-3, \
    0x1.9600000000000p+0, 0x1.db13db0d48000p-3, \
    0x1.9400000000000p+0, 0x1.e530effe72000p-3, \
    0x1.9000000000000p+0, 0x1.f991c6cb3c000p-3, \
    0x1.8e00000000000p+0, 0x1.01eae5626c000p-2, \
    0x1.8c00000000000p+0, 0x1.07138604d6000p-2, \
    0x1.8a00000000000p+0, 0x1.0c42d67616000p-2, \
    0x1.8800000000000p+0, 0x1.1178e8227e000p-2, \
    0x1.8400000000000p+0, 0x1.1bf99635a7000p-2, \
    0x1.8200000000000p+0, 0x1.214456d0ec000p-2, \
    0x1.8000000000000p+0, 0x1.269621134e000p-2, \
    0x1.7e00000000000p+0, 0x1.2bef07cdc9000p-2, \
    0x1.7c00000000000p+0, 0x1.314f1e1d36000p-2, \
    0x1.7a00000000000p+0, 0x1.36b6776be1000p-2, \
    0x1.7800000000000p+0, 0x1.3c25277333000p-2, \
    0x1.7600000000000p+0, 0x1.419b423d5f000p-2, \
    0x1.7400000000000p+0, 0x1.4718dc271c000p-2, \
    0x1.7200000000000p+0, 0x1.4c9e09e173000p-2, \
    0x1.7000000000000p+0, 0x1.522ae0738a000p-2, \
    0x1.6e00000000000p+0, 0x1.57bf753c8d000p-2, \
    0x1.6c00000000000p+0, 0x1.5d5bddf596000p-2, \
    0x1.6a00000000000p+0, 0x1.630030b3ab000p-2, \
    0x1.6800000000000p+0, 0x1.68ac83e9c7000p-2, \
    0x1.6600000000000p+0, 0x1.6e60ee6af2000p-2, \
    0x1.6400000000000p+0, 0x1.741d876c68000p-2, \
    0x1.6200000000000p+0, 0x1.79e26687d0000p-2, \
    0x1.6000000000000p+0, 0x1.7fafa3bd81000p-2, \
    0x1.5e00000000000p+0, 0x1.85855776dd000p-2, \
    0x1.5c00000000000p+0, 0x1.8b639a88b3000p-2, \
    0x1.5a00000000000p+0, 0x1.914a8635bf000p-2, \
    0x1.5800000000000p+0, 0x1.973a343135000p-2, \
    0x1.5600000000000p+0, 0x1.9d32bea15f000p-2, \
    0x1.5400000000000p+0, -0x1.22941fbcf8000p-2, \
    0x1.5300000000000p+0, -0x1.1f8ff9e48a000p-2, \
    0x1.5100000000000p+0, -0x1.1980d2dd42000p-2, \
    0x1.4f00000000000p+0, -0x1.136870293b000p-2, \
    0x1.4e00000000000p+0, -0x1.1058bf9ae5000p-2, \
    0x1.4c00000000000p+0, -0x1.0a324e2739000p-2, \
    0x1.4a00000000000p+0, -0x1.0402594b4d000p-2, \
    0x1.4900000000000p+0, -0x1.00e6c45ad5000p-2, \
    0x1.4700000000000p+0, -0x1.f550a564b8000p-3, \
    0x1.4500000000000p+0, -0x1.e8c0252aa6000p-3, \
    0x1.4400000000000p+0, -0x1.e27076e2b0000p-3, \
    0x1.4200000000000p+0, -0x1.d5c216b4fc000p-3, \
    0x1.4000000000000p+0, -0x1.c8ff7c79aa000p-3, \
    0x1.3f00000000000p+0, -0x1.c2968558c2000p-3, \
    0x1.3d00000000000p+0, -0x1.b5b519e8fc000p-3, \
    0x1.3c00000000000p+0, -0x1.af3c94e80c000p-3, \
    0x1.3a00000000000p+0, -0x1.a23bc1fe2c000p-3, \
    0x1.3900000000000p+0, -0x1.9bb362e7e0000p-3, \
    0x1.3700000000000p+0, -0x1.8e928de886000p-3, \
    0x1.3600000000000p+0, -0x1.87fa06520c000p-3, \
    0x1.3400000000000p+0, -0x1.7ab890210e000p-3, \
    0x1.3300000000000p+0, -0x1.740f8f5404000p-3, \
    0x1.3200000000000p+0, -0x1.6d60fe719e000p-3, \
    0x1.3000000000000p+0, -0x1.5ff3070a7a000p-3, \
    0x1.2f00000000000p+0, -0x1.59338d9982000p-3, \
    0x1.2d00000000000p+0, -0x1.4ba36f39a6000p-3, \
    0x1.2c00000000000p+0, -0x1.44d2b6ccb8000p-3, \
    0x1.2b00000000000p+0, -0x1.3dfc2b0ecc000p-3, \
    0x1.2900000000000p+0, -0x1.303d718e48000p-3, \
    0x1.2800000000000p+0, -0x1.29552f8200000p-3, \
    0x1.2700000000000p+0, -0x1.2266f190a6000p-3, \
    0x1.2500000000000p+0, -0x1.1478584674000p-3, \
    0x1.2400000000000p+0, -0x1.0d77e7cd08000p-3, \
    0x1.2300000000000p+0, -0x1.0671512ca6000p-3, \
    0x1.2100000000000p+0, -0x1.f0a30c0118000p-4, \
    0x1.2000000000000p+0, -0x1.e27076e2b0000p-4, \
    0x1.1f00000000000p+0, -0x1.d4313d66cc000p-4, \
    0x1.1e00000000000p+0, -0x1.c5e548f5bc000p-4, \
    0x1.1c00000000000p+0, -0x1.a926d3a4ac000p-4, \
    0x1.1b00000000000p+0, -0x1.9ab4246204000p-4, \
    0x1.1a00000000000p+0, -0x1.8c345d6318000p-4, \
    0x1.1900000000000p+0, -0x1.7da766d7b0000p-4, \
    0x1.1700000000000p+0, -0x1.60658a9374000p-4, \
    0x1.1600000000000p+0, -0x1.51b073f060000p-4, \
    0x1.1500000000000p+0, -0x1.42edcbea64000p-4, \
    0x1.1400000000000p+0, -0x1.341d7961bc000p-4, \
    0x1.1300000000000p+0, -0x1.253f62f0a0000p-4, \
    0x1.1200000000000p+0, -0x1.16536eea38000p-4, \
    0x1.1000000000000p+0, -0x1.f0a30c0118000p-5, \
    0x1.0f00000000000p+0, -0x1.d276b8adb0000p-5, \
    0x1.0e00000000000p+0, -0x1.b42dd71198000p-5, \
    0x1.0d00000000000p+0, -0x1.95c830ec90000p-5, \
    0x1.0c00000000000p+0, -0x1.77458f6330000p-5, \
    0x1.0b00000000000p+0, -0x1.58a5bafc90000p-5, \
    0x1.0a00000000000p+0, -0x1.39e87b9fe8000p-5, \
    0x1.0900000000000p+0, -0x1.1b0d989240000p-5, \
    0x1.0800000000000p+0, -0x1.f829b0e780000p-6, \
    0x1.0700000000000p+0, -0x1.b9fc027b00000p-6, \
    0x1.0600000000000p+0, -0x1.7b91b07d60000p-6, \
    0x1.0500000000000p+0, -0x1.3cea443470000p-6, \
    0x1.0400000000000p+0, -0x1.fc0a8b0fc0000p-7, \
    0x1.0300000000000p+0, -0x1.7dc475f820000p-7, \
    0x1.0200000000000p+0, -0x1.fe02a6b100000p-8, \
    0x1.0000000000000p+0, 0x0.0p+0, \
    0x0.0p+0, \
    0x1.4554412c584e0p-44, \
    0x1.98139928637fep-47, \
    -0x1.5439ce030a687p-44, \
    0x1.83e9ae021b67bp-45, \
    0x1.dac20827cca0cp-44, \
    0x1.9a19a8be97661p-44, \
    0x1.965c36e09f5fep-44, \
    -0x1.7e5dd7009902cp-46, \
    0x1.7a48ba8b1cb41p-44, \
    -0x1.19bd0ad125895p-44, \
    0x1.1cb7ce1d17171p-44, \
    -0x1.c0fe460d20041p-44, \
    0x1.3115c3abd47dap-45, \
    0x1.b1bdff50225c7p-44, \
    0x1.a89401fa71733p-46, \
    0x1.11fcba80cdd10p-44, \
    -0x1.7e5dd7009902cp-45, \
    0x1.1ef78ce2d07f2p-45, \
    0x1.00d238fd3df5cp-46, \
    0x1.39d6ccb81b4a1p-47, \
    0x1.19713c0cae559p-44, \
    -0x1.53e43558124c4p-44, \
    -0x1.27023eb68981cp-46, \
    -0x1.98c1d34f0f462p-44, \
    0x1.8e67be3dbaf3fp-44, \
    0x1.e0ddb9a631e83p-46, \
    -0x1.73d54aae92cd1p-47, \
    -0x1.337d94bcd3f43p-44, \
    -0x1.8724350562169p-45, \
    0x1.c794e562a63cbp-44, \
    0x1.ee138d3a69d43p-44, \
    -0x1.84a7e75b6f6e4p-47, \
    0x1.2806a847527e6p-44, \
    -0x1.fdbdbb13f7c18p-44, \
    -0x1.90d04cd7cc834p-44, \
    0x1.a43dcfade85aep-44, \
    -0x1.e76324e912b17p-44, \
    0x1.7188b163ceae9p-45, \
    0x1.1ef78ce2d07f2p-44, \
    -0x1.1ac89575c2125p-44, \
    -0x1.caf0428b728a3p-44, \
    -0x1.1b61f10522625p-44, \
    0x1.a9cfa4a5004f4p-45, \
    -0x1.8e27ad3213cb8p-45, \
    0x1.16ecdb0f177c8p-46, \
    0x1.83b54b606bd5cp-46, \
    -0x1.ce379226de3ecp-44, \
    0x1.06c18fb4c14c5p-44, \
    -0x1.e20891b0ad8a4p-45, \
    0x1.ebe708164c759p-45, \
    0x1.fadedee5d40efp-46, \
    -0x1.a0b2a08a465dcp-47, \
    -0x1.db623e731ae00p-45, \
    -0x1.7af966c548a30p-44, \
    -0x1.a37a6a0f7749ep-44, \
    -0x1.13a7b5b11cfa7p-44, \
    -0x1.309c168817444p-44, \
    0x1.46fb79bf6d4cbp-44, \
    -0x1.015486666443bp-44, \
    -0x1.05ae1e5e70470p-45, \
    0x1.a2652b44673e1p-44, \
    0x1.ab73b16bf4984p-44, \
    -0x1.6279e10d0c0b0p-45, \
    0x1.a6976f5eb0963p-44, \
    -0x1.7946c040cbe77p-45, \
    -0x1.b7b3a7a361c9ap-45, \
    0x1.d3e8499d67123p-44, \
    0x1.4ab9d817d52cdp-44, \
    -0x1.c6bee7ef4030ep-47, \
    -0x1.036b89ef42d7fp-48, \
    -0x1.cc68d52e01203p-50, \
    0x1.323e3a09202fep-45, \
    0x1.6805b80e8e6ffp-45, \
    0x1.a342c2af0003cp-44, \
    0x1.1ba91bbca681bp-45, \
    0x1.7794f689f8434p-45, \
    0x1.cfd73dee38a40p-45, \
    0x1.4b722ec011f31p-44, \
    0x1.a4e633fcd9066p-52, \
    0x1.539cd91dc9f0bp-44, \
    0x1.1f2a8a1ce0ffcp-45, \
    -0x1.a8154b13d72d5p-44, \
    -0x1.22120401202fcp-44, \
    0x1.bdb9072534a58p-45, \
    0x1.0b66c99018aa1p-44, \
    0x1.bc6e557134767p-44, \
    0x1.8586f183bebf2p-44, \
    -0x1.0ba68b7555d4ap-48, \
    0x1.4354bb3f219e5p-44, \
    0x1.70cc16135783cp-46, \
    -0x1.8a72a62b8c13fp-45, \
    0x1.680b5ce3ecb05p-50, \
    0x1.5b967f4471dfcp-44, \
    0x1.4d20ab840e7f6p-45, \
    -0x1.563451027c750p-46, \
    -0x1.cb2cd2ee2f482p-44, \
    0x1.a47579cdc0a3dp-45, \
    0x1.d599e83368e91p-44, \
    0x1.a342c2af0003cp-45, \
    0x1.9454379135713p-45, \
    -0x1.d0c57585fbe06p-46, \
    -0x1.563650bd22a9cp-44, \
    0x1.8a64826787061p-45, \
    -0x1.b20f5acb42a66p-44, \
    -0x1.2cc844480c89bp-44, \
    -0x1.0c3b1dee9c4f8p-44, \
    -0x1.83f69278e686ap-44, \
    -0x1.bc0eeea7c9acdp-46, \
    -0x1.1d09299837610p-44, \
    -0x1.416f8fb69a701p-44, \
    0x1.47c5e768fa309p-46, \
    0x1.d599e83368e91p-45, \
    -0x1.6a423c78a64b0p-46, \
    0x1.c827ae5d6704cp-46, \
    0x1.c148297c5feb8p-45, \
    0x1.181dce586af09p-44, \
    0x1.b2b739570ad39p-45, \
    -0x1.eafd480ad9015p-44, \
    0x1.3401e9ae889bbp-44, \
    -0x1.980267c7e09e4p-45, \
    0x1.b9a010ae6922ap-44, \
    0x1.3b955b602ace4p-44, \
    0x1.6a2c432d6a40bp-44, \
    -0x1.f1e7cf6d3a69cp-50, \
    0x1.eb1245b5da1f5p-44, \
    -0x1.9e23f0dda40e4p-46, \
    0x0.0p+0, \
    0x1.62e42fefa3800p-1, 0x1.ef35793c76730p-45, \
    0x1.239f4dd94c31bp-3, -0x1.555a2da07f467p-3, \
    0x1.99999cdd5fbafp-3, -0x1.fffffff9f41a8p-3, \
    0x1.5555555554472p-2, -0x1.0000000000005p-1, \
    0x1.45f306dc9c883p-1, 0x1.921fb54400000p+0, \
    0x1.0b4611a626330p-34, 0x1.45c06e0e68948p-86, \
    -0x1.ab17040cac9f2p-41, 0x1.61217daca8e8cp-33, \
    -0x1.ae6454110dacep-26, 0x1.71de3a545f9aap-19, \
    -0x1.a01a01a019930p-13, 0x1.1111111111110p-7, \
    -0x1.5555555555555p-3, -0x1.907cea09b716cp-37, \
    0x1.1eeb67ea7099fp-29, -0x1.27e4fa16e88e4p-22, \
    0x1.a01a019f4df8dp-16, -0x1.6c16c16c16964p-10, \
    0x1.5555555555555p-5, 0.0
template <class T>
PT_HD double log_tab(double x, T tab) {
    const T q = tab + MATH_LOG;
    const double m = frexp_mant(x);
    const int i = (int)(high_word(m) >> 13) & 127;
    const double k = (double)(frexp_exp(x) - 1 + (i >> 6));
    const double c = tab[2 * i], hi = tab[2 * i + 1], lo = tab[MATH_LO + i];
    const double r = fused(m, c, -1.0);
    const double w = fused(k, q[0], hi);  // exact: both parts end at 2^-42
    const double h = w + r;
    const double l = ((w - h) + r) + fused(k, q[1], lo);
    double p = fused(r, q[2], q[3]);
    p = fused(r, p, q[4]);
    p = fused(r, p, q[5]);
    p = fused(r, p, q[6]);
    p = fused(r, p, q[7]);
    return h + fused(r * r, p, l);
}

// sine and cosine of x in [0, 2 pi]: x = n pi/2 + y + t.  The first 33 bits of pi/2 times n
// subtract exactly, the next 50 bits times n are exact, and t is what y is rounded by with
// what is left of pi/2, so that y keeps its relative accuracy beside the multiples of pi/2
template <class T>
PT_HD void sincos_turn(double x, double& sn, double& cs, T tab) {
    const T q = tab + MATH_SIN;
    const double n = round_even(x * q[0]);
    const double a = fused(-n, q[1], x);
    const double w = n * q[2];
    const double y = a - w;
    const double t = fused(-n, q[3], (a - y) - w);
    const double z = y * y;
    double ps = fused(z, q[4], q[5]);
    ps = fused(z, ps, q[6]);
    ps = fused(z, ps, q[7]);
    ps = fused(z, ps, q[8]);
    ps = fused(z, ps, q[9]);
    ps = fused(z, ps, q[10]);
    double pc = fused(z, q[11], q[12]);
    pc = fused(z, pc, q[13]);
    pc = fused(z, pc, q[14]);
    pc = fused(z, pc, q[15]);
    pc = fused(z, pc, q[16]);
    const double hz = 0.5 * z, u = 1.0 - hz;
    const double s0 = y + fused(z * y, ps, t * u);
    // y^2 enters the cosine in first order: with what z was rounded by (and t)
    const double zt = fused(2.0 * t, y, fused(y, y, -z));
    const double c0 = u + (((1.0 - u) - hz) + fused(z * z, pc, -0.5 * zt));
    const int k = (int)n;
    const bool swap = (k & 1) != 0;
    sn = flip_sign(swap ? c0 : s0, (uint32_t)(k & 2) << 30);
    cs = flip_sign(swap ? s0 : c0, (uint32_t)((k + 1) & 2) << 30);
}

}  // namespace pt
