// exact_math.h -- arithmetic shortcuts that return exactly what the reference's FP32 operations
// return, shared by the HIP kernels and the host (so the CPU tests can check them exhaustively).
//
//  birp_div_rn(a, b, rb):   RN(a / b) for a precomputed rb = RN(1/b), by two residual corrections
//                           (q1 = q0 + (a - q0 b) rb is faithful; Markstein's theorem makes the
//                           second correction correctly rounded). Replaces the per-sample
//                           divisions of DataCube.cpp:206,209,212 and the ~12-instruction IEEE
//                           division sequence with 1 multiply + 4 FMAs.
//  birp_div_rn64(a, rb64):  RN(a / b) for rb64 = RN64(1/b): the float of the double product
//                           a * rb64. That product is within 2^-52 (relative) of a/b, while a
//                           quotient of two normal floats is never a float rounding midpoint and
//                           lies at least 2^-49 (relative) from every one (for a midpoint m,
//                           a - b m is a non-zero multiple of ulp(b) times half an ulp of the
//                           quotient, and b < 2^24 ulp(b)), so rounding the
//                           product to float gives RN(a/b) for every normal quotient. 3 VALU
//                           operations (two conversions and a double multiply).
//  birp_scale_sample(vw):   f32( f64(vw) * 637810000 / (4/pi) / 10000 ), the chain of
//                           Camera.cpp:201, as one double multiply by the chain's constant plus a
//                           guard: the two results differ by < 8 double ulps, so their float
//                           roundings agree unless the product lies within 16 double ulps of a
//                           float rounding midpoint (or outside the normal float range); those
//                           rare inputs take the three-operation chain.
//  birp_div_fma2(a, rh, rl): RN(a / b) for rh = RN(1/b) and rl = RN(1/b - rh), as one multiply and
//                           one FMA (Brisebarre, Muller and Raina, "Accelerating correctly rounded
//                           floating-point division when the divisor is known in advance", IEEE
//                           Trans. Computers 53(8), 2004). The sum a rh + RN(a rl) is within 2^-47
//                           (relative) of a/b, so it rounds like a/b for nearly every divisor; which
//                           ones is checked for all 2^23 significands of a when a cube is uploaded
//                           (the result does not depend on a's exponent or sign while a rl is a
//                           normal float), and the others keep birp_div_rn64.
//  birp_scale_fma2(vw):     the chain of Camera.cpp:201 the same way: the chain's constant as a sum of
//                           two floats, one multiply and one FMA. Equal to the chain for every
//                           significand of vw (checked exhaustively), while vw times the low part and
//                           the result are normal floats: |vw| in [2^-100, 2^110].
//  birp_sqrt_rn(a, y):      RN(sqrt(a)) for 2^-96 <= a, from an estimate y of 1 / sqrt(a) (a few ulps): one
//                           coupled step for the root and its half reciprocal, then the residual's
//                           correction (Markstein, "Computation of elementary functions on the IBM RISC
//                           System/6000 processor", IBM J. Res. Dev. 34(1), 1990), 7 operations. Checked for
//                           every significand of two binades with estimates off by up to 8 ulps.
//  birp_powf(b, e):         b^e for birp_powf_takes(b, e), in double: log2(b) = k + 2 atanh(s) / ln 2 with s =
//                           (m - 1) / (m + 1), m = b 2^-k in [sqrt(1/2), sqrt(2)), then 2^(e log2 b) from its
//                           fraction; minimax polynomials of 5 and 8 terms (Remez; 2^-39.7 absolute, 2^-34.5
//                           relative). The double's error is below 2^-33 for |e log2 b| < 64, so the result is
//                           the power's nearest float in all but one case of five hundred. 38 VALU operations
//                           (a double FMA issues like a float's here) for powf's 160.
//  birp_lerp_unit(a, b, t): std::lerp(a, b, t) for 0 <= t <= 1 - 2^-24 when a and b do not straddle
//                           zero: a + t (b - a), whose final clamp towards b never applies. Let
//                           X = RN(b - a) (b > a; the other case mirrors it), X = b - a + d with
//                           |d| <= ulp(X)/2. Since t <= 1 - 2^-24, RN(t X) <= X - ulp(X)/2 (a float;
//                           a subnormal X is exact, d = 0), so a + RN(t X) <= b + d - ulp(X)/2 <= b,
//                           and rounding keeps <= b. v_fract_f32 never returns more than 1 - 2^-24.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__) || defined(__HIP__)
#define BIRP_HD __host__ __device__ __forceinline__
#else
#include <math.h>
#include <string.h>
#define BIRP_HD static inline
#endif

#define BIRP_SCALE_K (1000 * 100 * 6378.1) /* 637810000.0 in double, as Camera.cpp:201 folds it */
#define BIRP_SCALE_C (4 / 3.14159265358979323846)

BIRP_HD float birp_fmaf(float a, float b, float c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_fmaf(a, b, c);
#else
    return fmaf(a, b, c);
#endif
}

BIRP_HD double birp_fma(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_fma(a, b, c);
#else
    return fma(a, b, c);
#endif
}

BIRP_HD uint32_t birp_f32_bits(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __float_as_uint(x);
#else
    uint32_t u;
    memcpy(&u, &x, sizeof(u));
    return u;
#endif
}
BIRP_HD float birp_f32_of(uint32_t u) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __uint_as_float(u);
#else
    float x;
    memcpy(&x, &u, sizeof(x));
    return x;
#endif
}

BIRP_HD uint64_t birp_f64_bits(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (uint64_t)__double_as_longlong(x);
#else
    uint64_t u;
    memcpy(&u, &x, sizeof(u));
    return u;
#endif
}

BIRP_HD float birp_div_rn(float a, float b, float rb) {
    float q0 = a * rb;
    float e0 = birp_fmaf(-q0, b, a);
    float q1 = birp_fmaf(e0, rb, q0);
    float e1 = birp_fmaf(-q1, b, a);
    return birp_fmaf(e1, rb, q1);
}

BIRP_HD float birp_div_rn64(float a, double rb64) { return (float)((double)a * rb64); }

BIRP_HD float birp_div_fma2(float a, float rh, float rl) { return birp_fmaf(a, rh, a * rl); }

BIRP_HD float birp_lerp_unit(float a, float b, float t) { return a + t * (b - a); }

BIRP_HD float birp_sqrt_rn(float a, float y) {
    float g = a * y, h = 0.5f * y;
    const float e = birp_fmaf(-h, g, 0.5f);
    g = birp_fmaf(g, e, g);
    h = birp_fmaf(h, e, h);
    return birp_fmaf(birp_fmaf(-g, g, a), h, g);
}

// The powers birp_powf takes: 2^-96 <= b < 2^96 and |e| < 2^20.
BIRP_HD int birp_powf_takes(float b, float e) {
    return birp_f32_bits(b) - 0x0F800000u < 0x60000000u && (birp_f32_bits(e) & 0x7FFFFFFFu) < 0x49800000u;
}

// A constant that stays in scalar registers beside its use: out of a loop the compiler would keep the
// polynomials' coefficients in 26 vector registers (the CMEM kernels' 77 became 101, 6 waves per SIMD 4).
BIRP_HD double birp_c64(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    int lo, hi;
    asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"(__double2loint(c)));
    asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"(__double2hiint(c)));
    return __hiloint2double(hi, lo);
#else
    return c;
#endif
}

BIRP_HD float birp_powf(float b, float e) {
    const uint32_t u = birp_f32_bits(b);
    const int k = (int)(u - 0x3F3504F3u) >> 23;
    const float m = birp_f32_of(u - ((uint32_t)k << 23));
    const double z = (double)(m - 1.0f), d = z + 2.0;  // exact
#if defined(__HIP_DEVICE_COMPILE__)
    double rc = (double)__builtin_amdgcn_rcpf(m + 1.0f);
#else
    double rc = (double)(1.0f / (m + 1.0f));
#endif
    rc = birp_fma(birp_fma(-d, rc, 1.0), rc, rc);
    const double s = z * rc, q = s * s;
    double p = birp_c64(0.34275912706533507);
    p = birp_fma(p, q, birp_c64(0.4115386565355376));
    p = birp_fma(p, q, birp_c64(0.577086533168229));
    p = birp_fma(p, q, birp_c64(0.9617966494089232));
    p = birp_fma(p, q, birp_c64(2.8853900818420084));
    const double t = (double)e * birp_fma(p, s, (double)k);
#if defined(__HIP_DEVICE_COMPILE__)
    const double n = __builtin_rint(t);
#else
    const double n = rint(t);
#endif
    const double f = t - n;
    p = birp_c64(1.5201923207590986e-05);
    p = birp_fma(p, f, birp_c64(0.00015469291175072532));
    p = birp_fma(p, f, birp_c64(0.0013333922556585357));
    p = birp_fma(p, f, birp_c64(0.009618027253562882));
    p = birp_fma(p, f, birp_c64(0.055504103534563094));
    p = birp_fma(p, f, birp_c64(0.24022651198158487));
    p = birp_fma(p, f, birp_c64(0.6931471807284448));
    p = birp_fma(p, f, birp_c64(0.9999999999616817));
#if defined(__HIP_DEVICE_COMPILE__)
    return (float)__builtin_amdgcn_ldexp(p, (int)n);
#else
    return (float)ldexp(p, (int)n);
#endif
}

// The reference chain, operation by operation (Camera.cpp:201).
BIRP_HD float birp_scale_chain(float vw) {
    return (float)(((double)vw * BIRP_SCALE_K / BIRP_SCALE_C) / 10000);
}

// The chain's constant: the chain applied to 1.0 (the first product is exact).
#define BIRP_SCALE_FOLDED ((1.0 * BIRP_SCALE_K / BIRP_SCALE_C) / 10000)

// The folded constant as a sum of two floats.
#define BIRP_SCALE_HI ((float)BIRP_SCALE_FOLDED)
#define BIRP_SCALE_LO ((float)(BIRP_SCALE_FOLDED - (double)BIRP_SCALE_HI))

BIRP_HD float birp_scale_fma2(float vw) { return birp_fmaf(vw, BIRP_SCALE_HI, vw * BIRP_SCALE_LO); }

// 1 when the folded product y cannot be trusted to round like the chain.
BIRP_HD int birp_scale_needs_chain(double y) {
    uint64_t u = birp_f64_bits(y);
    uint32_t lo = (uint32_t)u;
    uint32_t ex = (uint32_t)(u >> 52) & 0x7FFu;
    uint32_t m29 = lo & 0x1FFFFFFFu;
    int near_mid = (m29 - 0x0FFFFFF0u) < 0x21u;   /* |m29 - 2^28| <= 16 */
    int normal = (ex - 898u) <= 251u;             /* 2^-125 <= |y| < 2^127 */
    return (near_mid || !normal) && y != 0.0;
}

BIRP_HD float birp_scale_sample(float vw) {
    double y = (double)vw * BIRP_SCALE_FOLDED;
    if (birp_scale_needs_chain(y)) return birp_scale_chain(vw);
    return (float)y;
}
