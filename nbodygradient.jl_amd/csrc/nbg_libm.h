// nbg_libm.h -- portable FP64 elementary functions for the AHL21 step.
//
// One source, compiled both for gfx950 device code (hipcc) and for host code
// (g++), so that the GPU kernels and any CPU evaluation of the same formulas
// produce bit-identical results.  Every function is built only from IEEE
// operations that are exact or correctly rounded on both targets (+, -, *, /,
// sqrt, fma, rint, floor, frexp, ldexp) and must be compiled with
// -ffp-contract=off so no multiply-add is fused behind our back.
//
// Methods (all standard, published):
//  * sin/cos: Cody & Waite (1980) additive reduction by pi/2 with a three-part
//    constant (33+33+53 bits) for |x * 2/pi| < 2^20, Payne & Hanek (1983)
//    reduction with 2/pi to ~1330 bits above, then the Taylor series of sin and cos on
//    |r| <= pi/4 evaluated by Horner's rule in r^2, with the cos head
//    1 - r^2/2 evaluated in compensated form.
//  * exp: Cody & Waite reduction by ln 2 (32+53 bits), Taylor series of exp on
//    |r| <= ln2/2 to degree 13, exact scaling by 2^k with ldexp.
//  * sinh: odd Taylor series for |x| < 1, (e^x - e^-x)/2 above.
//  * cosh: (e^x + e^-x)/2.
//  * cbrt: exponent split with frexp, Halley iteration for the cube root of
//    the mantissa, ldexp back.
// Constants are generated by gen_libm_consts.py (mpmath, 200 digits).
//
// Accuracy (checked against libquadmath by the test suite): about 1 ulp over
// the full double range.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define NBG_HD __host__ __device__ inline
#else
#include <cmath>
#define NBG_HD inline
#endif

// Wave-uniform votes for device code: NBG_ALL(p) / NBG_ANY(p) are true when p
// holds on every / some active lane of the wave; on the host (one lane) both
// are p.  Device fast paths below are taken only when every active lane
// qualifies, so the branch is scalar and each lane's result is exactly what
// the general path would give it.
#if defined(__HIP_DEVICE_COMPILE__)
#define NBG_ALL(p) (__builtin_amdgcn_ballot_w64(!(p)) == 0)
#define NBG_ANY(p) (__builtin_amdgcn_ballot_w64((p)) != 0)
#else
#define NBG_ALL(p) (p)
#define NBG_ANY(p) (p)
#endif

// Rarely taken paths stay out of line in device code (one copy per kernel
// instead of one per call site).
#if defined(__HIP_DEVICE_COMPILE__)
#define NBG_HD_COLD NBG_HD __attribute__((noinline))
#else
#define NBG_HD_COLD NBG_HD
#endif

namespace nbg {

// Cody-Waite split of pi/2 and ln 2; 2/pi; log2(e).
constexpr double PIO2_1 = 0x1.921fb54400000p+0;
constexpr double PIO2_2 = 0x1.0b4611a600000p-34;
constexpr double PIO2_3 = 0x1.3198a2e037073p-69;
constexpr double TWO_OVER_PI = 0x1.45f306dc9c883p-1;
constexpr double LN2_1 = 0x1.62e42ff000000p-1;
constexpr double LN2_2 = -0x1.718432a1b0e26p-35;
constexpr double LOG2E = 0x1.71547652b82fep+0;
// 1/k! rounded to nearest double.
constexpr double F2 = 0x1.0000000000000p-1;
constexpr double F3 = 0x1.5555555555555p-3;
constexpr double F4 = 0x1.5555555555555p-5;
constexpr double F5 = 0x1.1111111111111p-7;
constexpr double F6 = 0x1.6c16c16c16c17p-10;
constexpr double F7 = 0x1.a01a01a01a01ap-13;
constexpr double F8 = 0x1.a01a01a01a01ap-16;
constexpr double F9 = 0x1.71de3a556c734p-19;
constexpr double F10 = 0x1.27e4fb7789f5cp-22;
constexpr double F11 = 0x1.ae64567f544e4p-26;
constexpr double F12 = 0x1.1eed8eff8d898p-29;
constexpr double F13 = 0x1.6124613a86d09p-33;
constexpr double F14 = 0x1.93974a8c07c9dp-37;
constexpr double F15 = 0x1.ae7f3e733b81fp-41;
constexpr double F16 = 0x1.ae7f3e733b81fp-45;
constexpr double F17 = 0x1.952c77030ad4ap-49;
constexpr double F18 = 0x1.6827863b97d97p-53;
constexpr double F19 = 0x1.2f49b46814157p-57;
constexpr double F21 = 0x1.71b8ef6dcf572p-66;

constexpr double EXP_OVF = 0x1.62e42fefa39efp+9;   // largest x with finite exp(x)
constexpr double EXP_UNF = -0x1.74910d52d3051p+9;  // below: exp(x) rounds to 0
constexpr double HUGE_D = 0x1.fffffffffffffp+1023;

NBG_HD double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a * b + c with c a constant: on the device the constant is taken from a
// scalar register pair by one v_fma_f64 (left to itself the compiler copies
// every 64-bit constant into vector registers with two moves per use).  The
// same fused multiply-add either way.
NBG_HD double fmac(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
#else
  return __builtin_fma(a, b, c);
#endif
}
// a / b and sqrt(x) for operands whose exponents are known to lie well inside
// the range (callers check |.| in [2^-250, 2^250], or a == 0 where the sign of
// a zero quotient does not matter): Newton's iteration on the hardware's
// approximate reciprocal (square root), then one correction by the exact
// remainder (Markstein 1990; Goldschmidt's coupled iteration for the root),
// which gives the correctly rounded result.  The compiler's own expansion adds
// exponent scaling and special-case fixes: 8 against 11 instructions and two
// waits for a quotient, 10 against 17 for a root.
NBG_HD double fdiv(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(b);
  r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
#else
  return a / b;
#endif
}
NBG_HD double fsqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
#else
  return __builtin_sqrt(x);
#endif
}
// a / b given r, 1 / b to about an ulp (the same correction).
NBG_HD double fdiv_by(double a, double b, double r) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
#else
  (void)r;
  return a / b;
#endif
}
// sqrt(x), and its reciprocal to about an ulp for fdiv_by: the iteration has it.
NBG_HD double fsqrt_recip(double x, double* r) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  const double q = h + h;
  *r = __builtin_fma(__builtin_fma(-g, q, 1.0), q, q);
  return g;
#else
  *r = 0.0;
  return __builtin_sqrt(x);
#endif
}
// a / c for a small positive whole number c, given rc = the double nearest to
// 1 / c: a * rc is within 1.5 ulp of the quotient, its remainder is exact, and
// the corrected quotient is within 2^-51 ulp of a / c before its one rounding,
// while a / c keeps at least 2^-15 ulp from every rounding boundary for
// c < 2^14 (a boundary times c needs more than 53 bits).  For a well inside
// the exponent range.
NBG_HD double cdiv(double a, double c, double rc) {
  const double q = a * rc;
  return __builtin_fma(__builtin_fma(-q, c, a), rc, q);
}
NBG_HD double rintd(double x) { return __builtin_rint(x); }
NBG_HD double fabsd(double x) { return __builtin_fabs(x); }
NBG_HD double copysignd(double a, double b) { return __builtin_copysign(a, b); }
NBG_HD double ldexpd(double x, int e) { return __builtin_ldexp(x, e); }
NBG_HD double frexpd(double x, int* e) { return __builtin_frexp(x, e); }
// the upper 32 bits of |x|: orders like |x| itself
NBG_HD int32_t hi_word(double x) { return (int32_t)((__builtin_bit_cast(uint64_t, x) >> 32) & 0x7fffffff); }
NBG_HD double infd() { return __builtin_inf(); }

// sin(hi + lo) on |hi| <= ~pi/4 (lo: tail of the reduced argument):
// hi - hi^3 * P(hi^2) + lo * (1 - hi^2/2), Taylor through hi^21.
NBG_HD double ksin(double hi, double lo) {
  const double z = hi * hi;
  double q = fmac(z, -F21, F19);
  q = fmac(z, q, -F17);
  q = fmac(z, q, F15);
  q = fmac(z, q, -F13);
  q = fmac(z, q, F11);
  q = fmac(z, q, -F9);
  q = fmac(z, q, F7);
  q = fmac(z, q, -F5);
  q = fmac(z, q, F3);
  // q = 1/3! - hi^2/5! + ...
  return hi + (lo * (1.0 - 0.5 * z) - (hi * z) * q);
}

// cos(hi + lo) on |hi| <= ~pi/4: 1 - hi^2/2 + hi^4 * Q(hi^2) - hi*lo, Taylor
// through hi^18, with the head 1 - hi^2/2 carried in compensated form.
NBG_HD double kcos(double hi, double lo) {
  const double z = hi * hi;
  double q = fmac(z, F18, -F16);
  q = fmac(z, q, F14);
  q = fmac(z, q, -F12);
  q = fmac(z, q, F10);
  q = fmac(z, q, -F8);
  q = fmac(z, q, F6);
  q = fmac(z, q, -F4);
  // q = -(1/4! - hi^2/6! + ...)
  const double hz = 0.5 * z;
  const double w = 1.0 - hz;
  return w + (((1.0 - w) - hz) - ((z * z) * q + hi * lo));
}

// 2/pi as 24 doubles c_i = M_i * 2^E_i (M_i of 53 bits in [1, 2), signed),
// each the nearest to 2/pi minus the ones before: their sum is 2/pi to
// about 2^-1330.  Mantissas and exponents are kept apart so that the tail,
// far below the double range, stays usable (gen_libm_consts.py).
struct Chunk {
  double m;
  int e;
};
constexpr Chunk TWO_OVER_PI_CHUNKS[24] = {
    {0x1.45f306dc9c883p+0, -1},     {-0x1.6b01ec5417056p+0, -55},   {-0x1.6447e493ad4cep+0, -109},
    {0x1.e21c820ff28b2p+0, -163},   {-0x1.508510ea79237p+0, -218},  {0x1.b8e909374b802p+0, -274},
    {-0x1.b6d115f62e6dep+0, -328},  {-0x1.80f10a71a76b3p+0, -383},  {0x1.cfba208d7d4bbp+0, -438},
    {-0x1.2edec598e3f65p+0, -494},  {-0x1.741037d8cdc54p+0, -549},  {0x1.cc1a99cfa4e42p+0, -603},
    {0x1.7e2ef7e4a0ec8p+0, -658},   {-0x1.da00087e99fc0p+0, -718},  {-0x1.0d0ee74a5f593p+0, -772},
    {0x1.f6d367ecf27cbp+0, -828},   {0x1.36e9e8c7ecd3dp+0, -885},   {-0x1.00ae9456c229cp+0, -939},
    {-0x1.41a0e84c2f8c6p+0, -996},  {-0x1.0eb5ada2b2809p+0, -1053}, {-0x1.0277039517bd5p+0, -1107},
    {0x1.98237e3db5d60p+0, -1167},  {-0x1.e6087beca1794p+0, -1221}, {0x1.da9e391615ee6p+0, -1276},
};
// pi/2 = PIO2_HI + PIO2_LO to about 2^-107.
constexpr double PIO2_HI = 0x1.921fb54442d18p+0;
constexpr double PIO2_LO = 0x1.1a62633145c07p-54;

// v mod 4 for |v| >= 4 (exact: v and 4 floor(v/4) are within a factor 2),
// v itself below.
NBG_HD double mod4(double v) { return fabsd(v) >= 4.0 ? v - 4.0 * __builtin_floor(v * 0.25) : v; }

// Payne & Hanek (1983) reduction for |x * 2/pi| >= 2^20, where the
// three-part Cody-Waite constant is no longer exact: x * 2/pi mod 4 from the
// exact products x * c_i (a product and its fma remainder), each reduced mod
// 4 exactly (Sterbenz) and summed with compensation (TwoSum); then
// r = x*2/pi - k with k the nearest integer, and x - k*pi/2 = r * pi/2 as
// hi + lo.  Products below 2^-131 are dropped (each later chunk is 2^-54
// smaller).  The rounding of the compensation term bounds the absolute error
// of the fraction by about 2^-94; the closest double to a multiple of pi/2,
// 6381956970095103 * 2^797, still comes out within 0.05 ulp.  Returns k mod 4.
NBG_HD_COLD int reduce_pio2_large(double x, double* hi, double* lo) {
  double sh = 0.0, sl = 0.0;
  for (int i = 0; i < 24; ++i) {
    const double xs = __builtin_ldexp(x, TWO_OVER_PI_CHUNKS[i].e);
    if (fabsd(xs) < 0x1p-132) break;  // this term and every later one are below 2^-130
    const double p = xs * TWO_OVER_PI_CHUNKS[i].m;
    const double e = __builtin_fma(xs, TWO_OVER_PI_CHUNKS[i].m, -p);  // x * c_i = p + e exactly
    const double terms[2] = {mod4(p), mod4(e)};
    for (int t = 0; t < 2; ++t) {  // (sh, sl) += term with TwoSum
      const double v = terms[t];
      const double s2 = sh + v;
      const double bv = s2 - sh;
      sl += (sh - (s2 - bv)) + (v - bv);
      sh = s2;
    }
  }
  const double k = rintd(sh);
  const double rh0 = sh - k;  // exact
  const double rh = rh0 + sl;
  const double rl = sl - (rh - rh0);
  const double yh = rh * PIO2_HI;
  const double yl = __builtin_fma(rh, PIO2_HI, -yh) + (rh * PIO2_LO + rl * PIO2_HI);
  *hi = yh + yl;
  *lo = yl - (*hi - yh);
  return (int)(k - 4.0 * __builtin_floor(k * 0.25));
}

// Simultaneous sine and cosine with one reduction.
NBG_HD void sincos(double x, double* s, double* c) {
#if defined(__HIP_DEVICE_COMPILE__)
  // Every active lane has 2^-27 <= |x| and rint(x * 2/pi) = 0: below, such a
  // lane takes the polynomial branch with hi = x, lo = +0 and quadrant 0.
  if (__all(fabsd(x * TWO_OVER_PI) < 0.5 && fabsd(x) >= 0x1p-27)) {
    *s = ksin(x, 0.0);
    *c = kcos(x, 0.0);
    return;
  }
#endif
  if (!(fabsd(x) <= HUGE_D)) {  // inf or nan
    *s = x - x;
    *c = x - x;
    return;
  }
  if (fabsd(x) < 0x1p-27) {  // sin x = x and cos x = 1 to within half an ulp
    *s = x;
    *c = 1.0;
    return;
  }
  const double k = rintd(x * TWO_OVER_PI);
  double hi, lo;
  int q;
  if (fabsd(k) < 0x1p20) {
    // x - k*pi/2 as hi + lo: k*PIO2_1 and k*PIO2_2 are exact for |k| < 2^20
    // and the first difference is exact (Sterbenz); the second is split with
    // Fast2Sum.
    const double t = x - k * PIO2_1;
    const double w = k * PIO2_2;
    const double r1 = t - w;
    const double e1 = (t - r1) - w;
    const double w3 = k * PIO2_3;
    hi = r1 - w3;
    lo = ((r1 - hi) - w3) + e1;
    const double kq = k - 4.0 * __builtin_floor(k * 0.25);  // k mod 4, exact
    q = (int)kq;
  } else {
    q = reduce_pio2_large(x, &hi, &lo);
  }
  const double sr = ksin(hi, lo);
  const double cr = kcos(hi, lo);
  switch (q) {
    case 0: *s = sr; *c = cr; break;
    case 1: *s = cr; *c = -sr; break;
    case 2: *s = -sr; *c = -cr; break;
    default: *s = -cr; *c = sr; break;
  }
}

NBG_HD double sin(double x) {
  double s, c;
  nbg::sincos(x, &s, &c);
  return s;
}

NBG_HD double cos(double x) {
  double s, c;
  nbg::sincos(x, &s, &c);
  return c;
}

// exp's Taylor polynomial on the reduced argument r
NBG_HD double exp_poly(double r) {
  double q = fmac(r, F13, F12);
  q = fmac(q, r, F11);
  q = fmac(q, r, F10);
  q = fmac(q, r, F9);
  q = fmac(q, r, F8);
  q = fmac(q, r, F7);
  q = fmac(q, r, F6);
  q = fmac(q, r, F5);
  q = fmac(q, r, F4);
  q = fmac(q, r, F3);
  q = fmac(q, r, F2);
  q = fmad(q, r, 1.0);
  return fmad(q, r, 1.0);
}

NBG_HD double exp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  // Every active lane has rint(x * log2 e) = 0 (so x is finite and in range):
  // below, such a lane reduces to r = x exactly and scales by 2^0.
  if (__all(fabsd(x * LOG2E) < 0.5)) return exp_poly(x);
#endif
  if (x != x) return x;
  if (x > EXP_OVF) return infd();
  if (x < EXP_UNF) return 0.0;
  const double k = rintd(x * LOG2E);
  const double r = (x - k * LN2_1) - k * LN2_2;
  double q = fmad(r, F13, F12);
  q = fmad(q, r, F11);
  q = fmad(q, r, F10);
  q = fmad(q, r, F9);
  q = fmad(q, r, F8);
  q = fmad(q, r, F7);
  q = fmad(q, r, F6);
  q = fmad(q, r, F5);
  q = fmad(q, r, F4);
  q = fmad(q, r, F3);
  q = fmad(q, r, F2);
  q = fmad(q, r, 1.0);
  const double p = fmad(q, r, 1.0);
  return ldexpd(p, (int)k);
}

// sinh's odd Taylor polynomial for |x| < 1
NBG_HD double sinh_poly(double x) {
  const double z = x * x;
  double q = fmac(z, F21, F19);
  q = fmac(q, z, F17);
  q = fmac(q, z, F15);
  q = fmac(q, z, F13);
  q = fmac(q, z, F11);
  q = fmac(q, z, F9);
  q = fmac(q, z, F7);
  q = fmac(q, z, F5);
  q = fmac(q, z, F3);
  return fmad(x * z, q, x);
}

NBG_HD double sinh(double x) {
  const double a = fabsd(x);
#if defined(__HIP_DEVICE_COMPILE__)
  if (__all(a < 1.0)) return sinh_poly(x);  // every active lane takes the branch below
#endif
  if (a < 1.0) {
    const double z = x * x;
    double q = fmad(z, F21, F19);
    q = fmad(q, z, F17);
    q = fmad(q, z, F15);
    q = fmad(q, z, F13);
    q = fmad(q, z, F11);
    q = fmad(q, z, F9);
    q = fmad(q, z, F7);
    q = fmad(q, z, F5);
    q = fmad(q, z, F3);
    return fmad(x * z, q, x);
  }
  if (x != x) return x;
  double y;
  if (a < 22.0) {
    const double e = nbg::exp(a);
    y = 0.5 * (e - 1.0 / e);
  } else if (a <= EXP_OVF) {
    y = 0.5 * nbg::exp(a);
  } else {
    const double h = nbg::exp(0.5 * a);
    y = (0.5 * h) * h;
  }
  return copysignd(y, x);
}

NBG_HD double cosh(double x) {
  const double a = fabsd(x);
  if (a != a) return a;
  if (a < 22.0) {
    const double e = nbg::exp(a);
    return 0.5 * (e + 1.0 / e);
  }
  if (a <= EXP_OVF) return 0.5 * nbg::exp(a);
  const double h = nbg::exp(0.5 * a);
  return (0.5 * h) * h;
}

// cube root of a finite nonzero x
NBG_HD double cbrt_core(double x) {
  int e;
  double m = frexpd(fabsd(x), &e);  // |x| = m * 2^e, m in [0.5, 1)
  int r = e % 3;
  if (r < 0) r += 3;
  m = ldexpd(m, r);  // m in [0.5, 4)
  e -= r;            // multiple of 3
  // minimax cubic on [0.5, 4), within 0.53 %; Halley's cubic convergence
  // (error -> 2/3 error^3) makes that 1e-7, then 1e-21
  double y = fmad(fmad(fmad(0x1.e14c60abbc5bep-7, m, -0x1.199a3aa9493a0p-3), m, 0x1.284527517da11p-1), m,
                  0x1.1504deb7050f6p-1);
  for (int it = 0; it < 2; ++it) {
    const double t = y * y * y;
    y = fdiv(y * (t + 2.0 * m), 2.0 * t + m);
  }
  // Newton polish with the residual y^3 - m evaluated in double-double.
  const double p = y * y;
  const double pe = fmad(y, y, -p);
  const double res = fmad(p, y, -m) + pe * y;
  y = y - fdiv(res, 3.0 * p);
  return copysignd(ldexpd(y, e / 3), x);
}

// cbrt_core for x in [2^-100, 2^100]: the device starts from the hardware's
// single-precision logarithm and exponential (within 3e-6, so one Halley step
// reaches 2e-17), 20 instructions against 60.  The polish's result is the
// cube root to about 2^-105 before its one rounding, so where it started from
// does not show.
NBG_HD double cbrt_mid(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)x) * 0.33333334f);
  const double t = y * y * y;
  y = fdiv(y * (t + 2.0 * x), 2.0 * t + x);
  const double p = y * y;
  const double pe = fmad(y, y, -p);
  const double res = fmad(p, y, -x) + pe * y;
  return y - fdiv(res, 3.0 * p);
#else
  return cbrt_core(x);
#endif
}

NBG_HD double cbrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (__all(x != 0.0 && fabsd(x) <= HUGE_D)) return cbrt_core(x);  // no lane needs the special case
#endif
  if (x == 0.0 || !(fabsd(x) <= HUGE_D)) return x + x;  // +-0, +-inf, nan
  return cbrt_core(x);
}

// Julia's sign(): -1, +1, or the (signed) zero / NaN itself.
NBG_HD double sign(double x) {
  return x < 0.0 ? -1.0 : (x > 0.0 ? 1.0 : x);
}

}  // namespace nbg
