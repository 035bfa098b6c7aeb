// crmath.h -- correctly rounded (with overwhelming probability) FP64 exp,
// log and pow, one source for the host (gcc, the oracle) and the device
// (hipcc, the FP64 kernels), so both evaluate them bit for bit alike.
//
// Method: Tang's table-driven algorithms (P. T. P. Tang, "Table-driven
// implementation of the exponential function", ACM TOMS 15(2), 1989, and
// "... of the logarithm function", ACM TOMS 16(4), 1990) carried in
// double-double arithmetic (Dekker's exact product by FMA, Knuth's
// two-sum), so that the value before the final rounding is within about
// 2^-70 of the true result; its one rounding to double is then the correct
// rounding except where the true value lies within that distance of a
// rounding boundary (a fraction of about 2^-17 of arguments).
//
//   log(x)   = k ln2 - log(invc_i) + log1p(r),  x = 2^k m, m in [1, 2),
//              i = the nearest of 1 + i/256 to m, invc_i = 1/(1 + i/256)
//              rounded, r = m invc_i - 1 formed exactly; log1p(r) by its
//              Taylor series to r^9 (|r| <= 2^-9)
//   exp(x)   = 2^e 2^(j/256) exp(r),  x = (256 e + j) ln2/256 + r,
//              |r| <= ln2/512; exp(r) by its Taylor series to r^7
//   pow(x,y) = exp(y log(x)) with log(x) and y log(x) as double-doubles
//
// Arguments outside the ranges the model produces (x <= 0, non-finite
// values, |result exponent| near the overflow range) are passed to the
// platform's own function.  The tables come from gen_crmath_tables.py.
#pragma once
#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define CRM_FN __host__ __device__ static inline
#define CRM_TABLE static constexpr
#else
#define CRM_FN static inline
#define CRM_TABLE static const
#endif

#include "crmath_tables.h"

CRM_FN uint64_t crm_bits(double x) {
  uint64_t u;
  __builtin_memcpy(&u, &x, 8);
  return u;
}
CRM_FN double crm_double(uint64_t u) {
  double x;
  __builtin_memcpy(&x, &u, 8);
  return x;
}
// s + e = a + b exactly (Knuth)
CRM_FN void crm_two_sum(double a, double b, double *s, double *e) {
  const double t = a + b, bb = t - a;
  *s = t;
  *e = (a - (t - bb)) + (b - bb);
}
// s + e = a + b exactly, |a| >= |b| or a = 0 (Dekker)
CRM_FN void crm_fast_two_sum(double a, double b, double *s, double *e) {
  const double t = a + b;
  *s = t;
  *e = b - (t - a);
}
// s + e = a + c b exactly, c b exact, |a| >= |c b| or a = 0
CRM_FN void crm_fast_two_sum_mul(double a, double c, double b, double *s, double *e) {
  const double t = __builtin_fma(c, b, a);
  *s = t;
  *e = __builtin_fma(c, b, a - t);
}
// p + e = a b exactly
CRM_FN void crm_two_prod(double a, double b, double *p, double *e) {
  const double t = a * b;
  *p = t;
  *e = __builtin_fma(a, b, -t);
}

// The main paths below are free of branches (whatever the argument, the table
// index is in range), so that several calls of one cell can be computed side
// by side: the waits of a call's two dependent table reads were the time of the
// kernels that make them.  An argument outside a main path's range takes the
// result of the *_rare function at the end.

// log(x 2^k0) as a double-double hi + lo, x positive and normal
CRM_FN void crm_log_dd(double x, int k0, double *hi, double *lo) {
  const uint64_t ix = crm_bits(x);
  // nearest table point 1 + i/256: the top nine mantissa bits, rounded; from
  // 1 + 511/512 up (i = 256) log(x) = (k+1) ln2 + log(m/2), m/2 near 1
  const int i = (int)(((ix >> 43) & 0x1ff) + 1) >> 1, wrap = i >> 8, j = i & (CRM_N - 1);
  const int k = (int)(ix >> 52) - 1023 + k0 + wrap;
  const double m = crm_double((ix & 0x000fffffffffffffULL) | ((uint64_t)(0x3ff - wrap) << 52));  // [1/2, 2)
  double p, e, rh, rl;
  crm_two_prod(m, CRM_LOG_INVC[j], &p, &e);
  crm_fast_two_sum(p - 1.0, e, &rh, &rl);  // p - 1 is exact (Sterbenz), a multiple of 2^-53, |e| <= 2^-54 below 1
  // log1p(rh + rl) = rh - rh^2/2 + rh^3/3 - ... + rl (1 - rh + rh^2) + ...
  double sh, sl;
  crm_two_prod(rh, rh, &sh, &sl);
  const double poly =
      rh * sh *
      (1. / 3. + rh * (-1. / 4. + rh * (1. / 5. + rh * (-1. / 6. + rh * (1. / 7. + rh * (-1. / 8. + rh * (1. / 9.)))))));
  double a, ea;
  crm_fast_two_sum_mul(rh, -0.5, sh, &a, &ea);
  const double l1 = ea + (rl + __builtin_fma(-0.5, sl, -(rh * rl) + (sh * rl + poly)));
  // k ln2 + T_j + a + l1: k LN2_HI is exact and 0 or above T_j, their sum 0 or above a
  const double kd = (double)k, T = CRM_LOG_T[2 * j];
  const double b = __builtin_fma(kd, CRM_LN2_HI, T), eb = T - __builtin_fma(-kd, CRM_LN2_HI, b);
  double c, ec;
  crm_fast_two_sum(b, a, &c, &ec);
  const double low = eb + ec + (kd * CRM_LN2_LO + CRM_LOG_T[2 * j + 1] + l1);
  crm_fast_two_sum(c, low, hi, lo);
}
CRM_FN int crm_log_main(double x) { return x >= 0x1p-1022 && x < __builtin_inf(); }
// log of a subnormal as a double-double
CRM_FN void crm_log_sub(double x, double *hi, double *lo) { crm_log_dd(x * 0x1p54, -54, hi, lo); }

CRM_FN double crm_log_rare(double x) {
  if (!(x > 0.) || x == __builtin_inf()) return log(x);
  double hi, lo;
  crm_log_sub(x, &hi, &lo);
  return hi + lo;
}
CRM_FN double crm_log(double x) {
  double hi, lo;
  crm_log_dd(x, 0, &hi, &lo);
  double r = hi + lo;
  if (__builtin_expect(!crm_log_main(x), 0)) r = crm_log_rare(x);
  return r;
}

// exp(xh + xl), |xl| <= ulp(xh), |xh| < 700
CRM_FN double crm_exp_dd(double xh, double xl) {
  // the nearest whole number, by adding it to the last place of 1.5 2^52
  const double kt = xh * CRM_INV_LN2N + 0x1.8p52, kd = kt - 0x1.8p52;
  const int k = (int)(uint32_t)crm_bits(kt);
  // r = xh + xl - k ln2/256, ln2/256 = C1 + C2 + C3
  double rh, rl;
  crm_two_sum(__builtin_fma(-kd, CRM_LN2N_C1, xh), -(kd * CRM_LN2N_C2), &rh, &rl);  // both products exact
  rl += xl - kd * CRM_LN2N_C3;
  crm_fast_two_sum(rh, rl, &rh, &rl);
  // expm1(rh + rl) = rh + rh^2/2 + rh^3/6 + ... + rl (1 + rh)
  double sh, sl;
  crm_two_prod(rh, rh, &sh, &sl);
  const double poly = rh * sh * (1. / 6. + rh * (1. / 24. + rh * (1. / 120. + rh * (1. / 720. + rh * (1. / 5040.)))));
  double a, ea;
  crm_fast_two_sum_mul(rh, 0.5, sh, &a, &ea);
  double ph, pl;
  crm_fast_two_sum(a, ea + (rl + __builtin_fma(0.5, sl, rh * rl + poly)), &ph, &pl);
  // 2^(j/256) (1 + p)
  const int j = k & (CRM_N - 1), e = k >> 8;
  const double th = CRM_EXP_T[2 * j], tl = CRM_EXP_T[2 * j + 1];
  double q1, q2, s, es;
  crm_two_prod(th, ph, &q1, &q2);
  crm_fast_two_sum(th, q1, &s, &es);
  const double r = s + (es + (q2 + (th * pl + (tl + tl * ph))));
  // times 2^e: exact for normal results (|e| <= 1010 here)
  return r * crm_double((uint64_t)(1023 + e) << 52);
}

CRM_FN double crm_exp(double x) {
  double r = crm_exp_dd(x, 0.);
  if (__builtin_expect(!(__builtin_fabs(x) < 700.), 0)) r = exp(x);
  return r;
}

// y (lh + ll) as a double-double
CRM_FN void crm_pow_arg(double lh, double ll, double y, double *zh, double *zl) {
  double h, l;
  crm_two_prod(y, lh, &h, &l);
  l += y * ll;
  crm_fast_two_sum(h, l, zh, zl);
}
CRM_FN double crm_pow_rare(double x, double y) {
  if (x == 1. || y == 0.) return 1.;
  if (!(x > 0.) || x == __builtin_inf() || !(__builtin_fabs(y) < __builtin_inf())) return pow(x, y);
  double lh, ll, zh, zl;
  if (x >= 0x1p-1022) crm_log_dd(x, 0, &lh, &ll);
  else crm_log_sub(x, &lh, &ll);
  crm_pow_arg(lh, ll, y, &zh, &zl);
  if (!(__builtin_fabs(zh) < 700.)) return pow(x, y);
  return crm_exp_dd(zh, zl);
}
CRM_FN double crm_pow(double x, double y) {
  double lh, ll, zh, zl;
  crm_log_dd(x, 0, &lh, &ll);
  crm_pow_arg(lh, ll, y, &zh, &zl);
  double r = crm_exp_dd(zh, zl);
  // (y infinite or NaN: zh is too)
  if (__builtin_expect(!(crm_log_main(x) && __builtin_fabs(zh) < 700.), 0)) r = crm_pow_rare(x, y);
  return r;
}

// two calls side by side
CRM_FN void crm_log2(double x0, double x1, double *r0, double *r1) {
  double h0, l0, h1, l1;
  crm_log_dd(x0, 0, &h0, &l0);
  crm_log_dd(x1, 0, &h1, &l1);
  double a = h0 + l0, b = h1 + l1;
  const int ok0 = crm_log_main(x0), ok1 = crm_log_main(x1);
  if (__builtin_expect(!(ok0 & ok1), 0)) {
    if (!ok0) a = crm_log_rare(x0);
    if (!ok1) b = crm_log_rare(x1);
  }
  *r0 = a;
  *r1 = b;
}
CRM_FN void crm_exp2(double x0, double x1, double *r0, double *r1) {
  double a = crm_exp_dd(x0, 0.), b = crm_exp_dd(x1, 0.);
  const int ok0 = __builtin_fabs(x0) < 700., ok1 = __builtin_fabs(x1) < 700.;
  if (__builtin_expect(!(ok0 & ok1), 0)) {
    if (!ok0) a = exp(x0);
    if (!ok1) b = exp(x1);
  }
  *r0 = a;
  *r1 = b;
}
CRM_FN void crm_pow2(double x0, double y0, double x1, double y1, double *r0, double *r1) {
  double lh, ll, z0, w0, z1, w1;
  crm_log_dd(x0, 0, &lh, &ll);
  crm_pow_arg(lh, ll, y0, &z0, &w0);
  crm_log_dd(x1, 0, &lh, &ll);
  crm_pow_arg(lh, ll, y1, &z1, &w1);
  double a = crm_exp_dd(z0, w0), b = crm_exp_dd(z1, w1);
  const int ok0 = crm_log_main(x0) & (__builtin_fabs(z0) < 700.), ok1 = crm_log_main(x1) & (__builtin_fabs(z1) < 700.);
  if (__builtin_expect(!(ok0 & ok1), 0)) {
    if (!ok0) a = crm_pow_rare(x0, y0);
    if (!ok1) b = crm_pow_rare(x1, y1);
  }
  *r0 = a;
  *r1 = b;
}
