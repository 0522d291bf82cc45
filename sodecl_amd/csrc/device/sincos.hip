// Sine and cosine of one argument for system sources: a call
// sincos(x, &s, &c) in the plugin resolves to sodecl_sincos unless the caller
// asks for the device library's.  Like sin.hip the file is also valid host C++
// (define SODECL_MATH_FN first; it follows sin.hip, whose helpers it uses), so
// that the same operations can be checked on the CPU.
//
// Method: q = round(x 2/pi) by one fused multiply-add with 1.5 2^52 (the sum's
// low word is q mod 2^32, two's complement), and r = x - q pi/2 by Cody and
// Waite's additive reduction (W. J. Cody, W. Waite, "Software Manual for the
// Elementary Functions", 1980) with pi/2 = P1 + P2 (|pi/2 - P1 - P2| <
// 1.5e-33): r1 = x - q P1 is exact (both terms are multiples of 2^-53 while
// |x| < 1 and of 2^-52 from there on, |r1| < 1), r = r1 - q P2 rounds and
// t = (r1 - r) - q P2 is that rounding.  On |r| <= pi/4, z = r^2:
//   sin(r + t) = r + (r^3 S(z) + t (1 - z/2)),
//   cos(r + t) = w + (((1 - w) - z/2) + (z^2 C(z) - t r)),  w = round(1 - z/2),
// S and C of degree 5 within 2.1e-17 of (sin r - r)/r^3 and 1.3e-18 of
// (cos r - 1 + z/2)/r^4 (sincos_coefficients.py derives every constant).
// Everything but the leading term is at most 0.12 of the sine and 0.04 of the
// cosine, so its roundings stay small: at most 0.83 ulp for either one
// measured on 2.1e7 arguments up to 1e9.
// The device library's sincos is used for |x| > 2^30 (and NaN, infinities),
// for zeros (whose sign the sums above lose), and within 4 |q| P2 of a nonzero multiple of pi/2, where the two-double
// pi/2 is too short for the relative accuracy of the smaller result.
//
// Cost on gfx950: 45 VALU instructions and five for the range test, against
// about 60 for the noise's sodecl_sincos_reduced, which keeps the products'
// rounding errors as well (0.58 ulp).

#ifndef SODECL_MATH_FN
#define SODECL_MATH_FN __host__ __device__ inline
#endif

#if defined(__clang__)
#define SODECL_SINCOS_NO_CONTRACT _Pragma("clang fp contract(off)")
#else
#define SODECL_SINCOS_NO_CONTRACT
#endif

// sin x and cos x by the reduction above; false where it does not hold.
SODECL_MATH_FN bool sodecl_sincos_core(double x, double* sx, double* cx)
{
    SODECL_SINCOS_NO_CONTRACT
    const double p2 = 0x1.1a62633145c07p-54;
    const double kk = sodecl_fma_k(x, 0x1.45f306dc9c883p-1, 0x1.8p52);
    const double q = kk - 0x1.8p52;
    const double r1 = fma(-q, 0x1.921fb54442d18p+0, x);
    const double r = fma(-q, p2, r1);
    const double t = fma(-q, p2, r1 - r);
    const double z = r * r;
    double sp = 0x1.5e0b05bff20f2p-33;
    sp = sodecl_fma_k(sp, z, -0x1.ae600aca92c64p-26);
    sp = sodecl_fma_k(sp, z, 0x1.71de379654304p-19);
    sp = sodecl_fma_k(sp, z, -0x1.a01a019e83816p-13);
    sp = sodecl_fma_k(sp, z, 0x1.1111111110bb2p-7);
    sp = sodecl_fma_k(sp, z, -0x1.5555555555555p-3);
    double cp = -0x1.907d8f29fe831p-37;
    cp = sodecl_fma_k(cp, z, 0x1.1eeb68cd22f56p-29);
    cp = sodecl_fma_k(cp, z, -0x1.27e4fa17bf139p-22);
    cp = sodecl_fma_k(cp, z, 0x1.a01a019f4e9b4p-16);
    cp = sodecl_fma_k(cp, z, -0x1.6c16c16c16967p-10);
    cp = sodecl_fma_k(cp, z, 0x1.5555555555555p-5);
    const double w = fma(z, -0.5, 1.0);
    const double sin_r = r + fma(z * r, sp, t * w);
    const double cos_r = w + fma(z * z, cp, fma(-t, r, fma(z, -0.5, 1.0 - w)));
    // quadrant: sin x = +-sin r or +-cos r, cos x = +-cos r or +-sin r
    unsigned n;   // low word of kk (little-endian on the host and the GPU)
    __builtin_memcpy(&n, &kk, sizeof n);
    const double a = (n & 1u) ? cos_r : sin_r;
    const double b = (n & 1u) ? sin_r : cos_r;
    *sx = sodecl_with_hi_word(a, sodecl_hi_word(a) ^ ((n & 2u) << 30));
    *cx = sodecl_with_hi_word(b, sodecl_hi_word(b) ^ (((n + 1u) & 2u) << 30));
    return fabs(x) <= 0x1p30 && fabs(r) > fabs(q) * (4.0 * p2);
}

SODECL_MATH_FN void sodecl_sincos(double x, double* s, double* c)
{
    if (__builtin_expect(!sodecl_sincos_core(x, s, c), 0)) sincos(x, s, c);
}
SODECL_MATH_FN void sodecl_sincos(float x, float* s, float* c) { sincosf(x, s, c); }

// The same with NaN as the sine where the library's function is needed, for
// sources that carry it to a sum (SODE_FIELD_MARKED_SINCOS): the caller tests
// many arguments at once (field.hip).  A mark on the cosine as well costs 1 to
// 2.5% of the field kernels (1500 orbits of 33 components 351 -> 360 us).
SODECL_MATH_FN void sodecl_sincos_marked(double x, double* s, double* c)
{
    if (!sodecl_sincos_core(x, s, c)) *s = sodecl_with_hi_word(*s, 0x7ff80000u);
}
SODECL_MATH_FN void sodecl_sincos_marked(float x, float* s, float* c) { sincosf(x, s, c); }
