// xmath.hpp - x^y in FP64 as exp(y ln x) with short polynomials.
//
// The flux functions raise positive reals to non-integer powers (van
// Genuchten retention and conductivity, Manning's depth^(2/3), channel
// geometry) about seven times per element per call.  The device library's
// pow carries a double-double logarithm and full special-case handling
// (some 215 VALU instructions); this one is about 65:
//
//   ln x:   x = m 2^e with m in [sqrt(1/2), sqrt(2)),  f = (m-1)/(m+1),
//           ln m = 2 atanh f = 2f (1 + f^2/3 + f^4/5 + ... + f^18/21)
//           (|f| <= 0.1716, the first omitted term is below 2^-56), and
//           ln x = e ln2_hi + (e ln2_lo + ln m) kept as a hi + lo pair
//           (ln2 split as in Cody and Waite, ln2_hi exact in 32 bits).
//   t:      y ln x = thi + tlo with the product's rounding error from fma.
//   exp t:  k = rint(thi / ln2),  r = (thi - k ln2_hi) + (tlo - k ln2_lo)
//           (|r| <= ln2 / 2), exp r by its Taylor series to r^13/13!
//           (remainder below 2^-57), scaled by 2^k.
//
// Error: t carries about |y| 1.2e-16 absolute error, exp about 1 ulp, so x^y
// is within a few ulp of the exact power for the exponents used here
// (|y| <= 3); the unit tests measure it against the host libm's pow.
// Exact where the reference's results are exact and the formulas depend on
// it: 1^y = 1, 0^y = +0 for y > 0, and x^y >= 1 for x >= 1, y >= 0 (so
// pow(1/s, m) - 1 never goes negative).  Zero, negative and non-finite
// arguments follow C's pow.  Nothing here is a call: a call in the element
// path of the RHS kernels made the compiler keep every kernel argument that
// lives across it in vector lanes (900 v_readlane in the one-launch RHS).
//
// Host and device compile the same operations (explicit fma, no
// contraction), so both return the same bits.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace pihm {

#define PIHM_HD __host__ __device__ __forceinline__

// A coefficient of a device polynomial, held in a scalar register pair: p =
// fma(p, s, c) is then one vector instruction that reads c from the scalar
// file, and K polynomials in step share it.  Left to itself the compiler copies
// c into the vector register that the multiply-add overwrites, two more vector
// instructions for each term.
PIHM_HD double coef(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(c));
#endif
  return c;
}

constexpr double kLn2Hi = 6.93147180369123816490e-01;  // 0x3FE62E42FEE00000: 32 significant bits
constexpr double kLn2Lo = 1.90821492927058770002e-10;  // ln 2 - kLn2Hi

// x = m 2^e with m in [1/2, 1), for finite x > 0.
PIHM_HD double split_exp(double x, int *e) {
#if defined(__HIP_DEVICE_COMPILE__)
  *e = __builtin_amdgcn_frexp_exp(x);
  return __builtin_amdgcn_frexp_mant(x);
#else
  return frexp(x, e);
#endif
}

// (m - 1) / (m + 1) for m in [1/2, 2): on the device a reciprocal refined to
// full precision, the quotient and its exact remainder (Markstein), without
// the scaling and special cases of a general division that no such m needs.
PIHM_HD double log_ratio(double m) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double n = m - 1.0, d = m + 1.0;       // n is exact
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return fma(fma(-d, q, n), r, q);
#else
  return (m - 1.0) / (m + 1.0);
#endif
}

// Division with the reciprocal apart, so that quotients by one divisor share
// it: the operations of the compiler's own division (the hardware estimate,
// two Newton steps, the quotient corrected by its exact remainder, the special
// cases) without its scaling, which only operands near the ends of the range
// of a double need.  Correctly rounded, as the host's division, elsewhere.
// 52 cycles a wavefront (75 with the scaling), 18 for each further quotient.
struct Recip {
  double b, r;
};
PIHM_HD Recip recip_of(double b) {
  Recip R{b, 0.0};
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(b);
  r = fma(fma(-b, r, 1.0), r, r);
  R.r = fma(fma(-b, r, 1.0), r, r);
#endif
  return R;
}
PIHM_HD double quot(double a, const Recip &R) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double q = a * R.r;
  return __builtin_amdgcn_div_fixup(fma(fma(-R.b, q, a), R.r, q), R.b, a);
#else
  return a / R.b;
#endif
}
PIHM_HD double fdiv(double a, double b) { return quot(a, recip_of(b)); }

// sqrt(x), the same way: the compiler's sequence (hardware estimate,
// Goldschmidt, two corrections by the exact remainder) without the scaling that
// x below 2^-767 needs.  56 cycles a wavefront instead of 105.  x > 0 finite.
PIHM_HD double sqrt_mid(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
#else
  return sqrt(x);
#endif
}
// The same for any x >= 0 (zero and infinity; NaN passes through).
PIHM_HD double sqrt_pos(double x) {
  const double g = sqrt_mid(x);
  return (x > 0.0 && x < HUGE_VAL) ? g : x;
}

// The logarithm and the exponential work on K arguments in step, so that one
// wavefront has K independent chains of multiply-adds in flight; each
// argument's arithmetic is the same for every K.

// ln x = hi + lo for finite x > 0 (normal or subnormal); the pair carries
// ln x to about 1.2e-16 absolute whatever the exponent of x.
template <int K>
PIHM_HD void ln_pos_n(const double (&x)[K], double (&hi)[K], double (&lo)[K]) {
  double f[K], s[K], p[K], de[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    int e;
    double m = split_exp(x[k], &e);                // x = m 2^e, m in [1/2, 1)
    if (m < 0.70710678118654752440) {
      m = m + m;
      e -= 1;
    }
    f[k] = log_ratio(m);
    s[k] = f[k] * f[k];
    de[k] = (double)e;
  }
#define PIHM_STEP(c) { const double cc = coef(c); for (int k = 0; k < K; k++) p[k] = fma(p[k], s[k], cc); }
  { const double cc = coef(1.0 / 21.0); for (int k = 0; k < K; k++) p[k] = cc; }
  PIHM_STEP(1.0 / 19.0) PIHM_STEP(1.0 / 17.0) PIHM_STEP(1.0 / 15.0) PIHM_STEP(1.0 / 13.0) PIHM_STEP(1.0 / 11.0)
  PIHM_STEP(1.0 / 9.0) PIHM_STEP(1.0 / 7.0) PIHM_STEP(1.0 / 5.0) PIHM_STEP(1.0 / 3.0)
#undef PIHM_STEP
#pragma unroll
  for (int k = 0; k < K; k++) {
    const double f2 = f[k] + f[k];
    const double lnm = fma(f2 * s[k], p[k], f2);   // |lnm| <= 0.35
    const double a = de[k] * kLn2Hi;               // exact: |e| < 2^11
    const double b = fma(de[k], kLn2Lo, lnm);
    hi[k] = a + b;                                 // |a| >= |b| unless a == 0
    lo[k] = (a - hi[k]) + b;
  }
}

// e^(hi + lo) for |hi| < 1000 and |lo| <= ulp(hi): past the range of a double
// the final scaling gives infinity, a subnormal or zero.
template <int K>
PIHM_HD void exp_core_n(const double (&hi)[K], const double (&lo)[K], double (&out)[K]) {
  double kk[K], r[K], p[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    kk[k] = rint(hi[k] * 1.44269504088896340736);
    r[k] = fma(-kk[k], kLn2Hi, hi[k]);             // exact for |kk| < 2^21
    r[k] = r[k] + fma(-kk[k], kLn2Lo, lo[k]);      // |r| <= ln2 / 2 + 1e-10
  }
#define PIHM_STEP(c) { const double cc = coef(c); for (int k = 0; k < K; k++) p[k] = fma(p[k], r[k], cc); }
  { const double cc = coef(1.0 / 6227020800.0); for (int k = 0; k < K; k++) p[k] = cc; }   // 1/13!
  PIHM_STEP(1.0 / 479001600.0) PIHM_STEP(1.0 / 39916800.0) PIHM_STEP(1.0 / 3628800.0) PIHM_STEP(1.0 / 362880.0)
  PIHM_STEP(1.0 / 40320.0) PIHM_STEP(1.0 / 5040.0) PIHM_STEP(1.0 / 720.0) PIHM_STEP(1.0 / 120.0)
  PIHM_STEP(1.0 / 24.0) PIHM_STEP(1.0 / 6.0)
#undef PIHM_STEP
#pragma unroll
  for (int k = 0; k < K; k++) {
    p[k] = fma(p[k], r[k], 0.5);
    p[k] = fma(p[k], r[k], 1.0);
    p[k] = fma(p[k], r[k], 1.0);
    out[k] = ldexp(p[k], (int)kk[k]);
  }
}

PIHM_HD double ln_pos(double x, double *lo) {
  const double xs[1] = {x};
  double h[1], l[1];
  ln_pos_n<1>(xs, h, l);
  *lo = l[0];
  return h[0];
}
PIHM_HD double exp_core(double hi, double lo) {
  const double h[1] = {hi}, l[1] = {lo};
  double r[1];
  exp_core_n<1>(h, l, r);
  return r[0];
}

// e^(hi + lo) for any hi (the pair as above).
PIHM_HD double exp_pair(double hi, double lo) {
  if (fabs(hi) < 1000.0) return exp_core(hi, lo);
  return hi > 0.0 ? HUGE_VAL : (hi < 0.0 ? 0.0 : hi);   // the last: NaN
}

// y (hi + lo) as a pair.
PIHM_HD double mul_pair(double y, double hi, double lo, double *tlo) {
  const double thi = y * hi;
  *tlo = fma(y, hi, -thi) + y * lo;
  return thi;
}

// x^y of the arguments xpow's main path does not take (C's pow, Annex F).
// For a negative x and an integer y it sets *ax = |x| and *neg (y odd)
// instead: the main path evaluates (*ax)^y.
PIHM_HD double pow_special(double x, double y, double *ax, bool *neg) {
  const double a = fabs(x);
  const bool odd = rint(y) == y && rint(0.5 * y) != 0.5 * y;
  if (y == 0.0 || x == 1.0) return 1.0;
  if (isnan(x) || isnan(y)) return x + y;
  if (a == 0.0 || a == HUGE_VAL) {
    const double r = ((a == 0.0) == (y > 0.0)) ? 0.0 : HUGE_VAL;
    return (odd && signbit(x)) ? -r : r;
  }
  if (fabs(y) == HUGE_VAL) return (a == 1.0) ? 1.0 : (((a > 1.0) == (y > 0.0)) ? HUGE_VAL : 0.0);
  if (rint(y) != y) return NAN;    // finite x < 0, y not an integer
  *ax = a;
  *neg = odd;
  return 0.0;
}

// x^y: finite x > 0 and finite y; (+0)^y = +0 for y > 0; the rest as
// pow_special says.
PIHM_HD double xpow(double x, double y) {
  double ax = x, r = 0.0;
  bool neg = false, main_path = x > 0.0 && x < HUGE_VAL && fabs(y) < HUGE_VAL;
  if (!main_path && !(x == 0.0 && y > 0.0 && !signbit(x))) {
    ax = 0.0;
    r = pow_special(x, y, &ax, &neg);
    main_path = ax > 0.0;
  }
  if (main_path) {
    double lo, tlo;
    const double hi = ln_pos(ax, &lo);
    const double thi = mul_pair(y, hi, lo, &tlo);
    r = exp_pair(thi, tlo);
    if (neg) r = -r;
  }
  return r;
}

// x[k]^y[k] for x >= 0 and y > 0 with |y ln x| < 1000, K powers in step and no
// branch: xpow's value for each (0^y = 0, infinity and NaN pass through).
template <int K>
PIHM_HD void xpow_n(const double (&x)[K], const double (&y)[K], double (&r)[K]) {
  double xx[K], hi[K], lo[K], th[K], tl[K];
#pragma unroll
  for (int k = 0; k < K; k++) xx[k] = (x[k] > 0.0 && x[k] < HUGE_VAL) ? x[k] : 1.0;
  ln_pos_n<K>(xx, hi, lo);
#pragma unroll
  for (int k = 0; k < K; k++) th[k] = mul_pair(y[k], hi[k], lo[k], &tl[k]);
  exp_core_n<K>(th, tl, r);
#pragma unroll
  for (int k = 0; k < K; k++) r[k] = (x[k] > 0.0 && x[k] < HUGE_VAL) ? r[k] : x[k];
}

// ---------------------------------------------------------------------------
// The same two functions as the device library has them, to a little over half
// an ulp, for the land-surface step, whose powers and logarithms were the
// library's: what the short ones above leave out, the rounding of the
// logarithm's quotient and of the exponential's sums, is carried along (some
// 15 operations more for a power).

// ln x = hi + lo for finite x > 0, the pair to about 3e-18 of its size.
template <int K>
PIHM_HD void ln_fine_n(const double (&x)[K], double (&hi)[K], double (&lo)[K]) {
  double q[K], ql[K], s[K], p[K], de[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    int e;
    double m = split_exp(x[k], &e);
    if (m < 0.70710678118654752440) {
      m = m + m;
      e -= 1;
    }
    const double n = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);   // n is exact, d + dl = m + 1
    q[k] = log_ratio(m);                                         // n / d, rounded
    // the rest of n / (d + dl); 1 / (m + 1) is (1 - q) / 2 as well as it needs to be
    ql[k] = fma(-q[k], dl, fma(-q[k], d, n)) * fma(-0.5, q[k], 0.5);
    s[k] = q[k] * q[k];
    de[k] = (double)e;
  }
#define PIHM_STEP(c) { const double cc = coef(c); for (int k = 0; k < K; k++) p[k] = fma(p[k], s[k], cc); }
  { const double cc = coef(1.0 / 21.0); for (int k = 0; k < K; k++) p[k] = cc; }
  PIHM_STEP(1.0 / 19.0) PIHM_STEP(1.0 / 17.0) PIHM_STEP(1.0 / 15.0) PIHM_STEP(1.0 / 13.0) PIHM_STEP(1.0 / 11.0)
  PIHM_STEP(1.0 / 9.0) PIHM_STEP(1.0 / 7.0) PIHM_STEP(1.0 / 5.0) PIHM_STEP(1.0 / 3.0)
#undef PIHM_STEP
#pragma unroll
  for (int k = 0; k < K; k++) {
    const double f2 = q[k] + q[k], fl = ql[k] + ql[k];
    // beyond 2 q: the series' other terms, at most a hundredth of it, and ql's share 2 ql / (1 - s)
    const double t = fma(f2 * s[k], p[k], fma(fl, s[k], fl));
    const double a = de[k] * kLn2Hi;               // exact
    const double h = a + f2, l = (a - h) + f2;     // exact: |a| >= |f2| or a == 0
    const double r = l + fma(de[k], kLn2Lo, t);
    hi[k] = h + r;
    lo[k] = (h - hi[k]) + r;
  }
}

// e^(hi + lo) for any hi, |lo| <= ulp(hi).
PIHM_HD double exp_fine(double hi, double lo) {
  if (!(fabs(hi) < 1000.0)) return hi > 0.0 ? HUGE_VAL : (hi < 0.0 ? 0.0 : hi);   // the last: NaN
  const double kk = rint(hi * 1.44269504088896340736);
  const double r0 = fma(-kk, kLn2Hi, hi);          // exact
  double rl = fma(-kk, kLn2Lo, lo);
  const double r = r0 + rl;                        // |r| <= ln2 / 2 + 1e-10
  rl = (r0 - r) + rl;
  double p = coef(1.0 / 6227020800.0);
#define PIHM_STEP(c) p = fma(p, r, coef(c));
  PIHM_STEP(1.0 / 479001600.0) PIHM_STEP(1.0 / 39916800.0) PIHM_STEP(1.0 / 3628800.0) PIHM_STEP(1.0 / 362880.0)
  PIHM_STEP(1.0 / 40320.0) PIHM_STEP(1.0 / 5040.0) PIHM_STEP(1.0 / 720.0) PIHM_STEP(1.0 / 120.0)
  PIHM_STEP(1.0 / 24.0) PIHM_STEP(1.0 / 6.0)
#undef PIHM_STEP
  const double h = 1.0 + r, l = (1.0 - h) + r;     // exact
  const double u = fma(rl, h, (r * r) * fma(p, r, 0.5));
  return ldexp(h + (l + u), (int)kk);
}

// ln x for any x.
PIHM_HD double ln_fine(double x) {
  if (x > 0.0 && x < HUGE_VAL) {
    const double xs[1] = {x};
    double h[1], l[1];
    ln_fine_n<1>(xs, h, l);
    return h[0];                                   // h + l rounded
  }
  return (x == 0.0) ? -HUGE_VAL : ((x < 0.0) ? NAN : x);
}

// x^y as the C library's, special arguments included.
PIHM_HD double pow_fine(double x, double y) {
  double ax = x, r = 0.0;
  bool neg = false, main_path = x > 0.0 && x < HUGE_VAL && fabs(y) < HUGE_VAL;
  if (!main_path && !(x == 0.0 && y > 0.0 && !signbit(x))) {
    ax = 0.0;
    r = pow_special(x, y, &ax, &neg);
    main_path = ax > 0.0;
  }
  if (main_path) {
    const double xs[1] = {ax};
    double h[1], l[1], tlo;
    ln_fine_n<1>(xs, h, l);
    const double thi = mul_pair(y, h[0], l[0], &tlo);
    r = exp_fine(thi, tlo);
    if (neg) r = -r;
  }
  return r;
}

// x^3 and x^4, a rounding apart from the exact product's rounding.
PIHM_HD double cube(double x) {
  const double s = x * x, c = s * x;
  return c + fma(fma(x, x, -s), x, fma(s, x, -c));
}
PIHM_HD double fourth(double x) {
  const double s = x * x, q = s * s;
  return q + fma(2.0 * s, fma(x, x, -s), fma(s, s, -q));
}

}  // namespace pihm
