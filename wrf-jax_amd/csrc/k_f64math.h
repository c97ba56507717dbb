// Natural logarithm and power in FP64: f64_log and f64_pow for results that are
// rounded once to FP32 (calc_p_rho_phi's log(pfd / pfu) and temp^(cp/cv)),
// f64_pow_full for results that stay in FP64 (the energy of wrfdc_checksums).
//
// Written from the series, not a vendor library: the device library's FP64
// log and pow are full FP64-accuracy routines (extra-precision logarithm
// inside pow) and made the kernel that calls them bound by vector ALU issue.
// An FP64 result within a few ulp of the true value already rounds to the
// same FP32 value as a correctly rounded one except when the true value
// lies within ~1e-15 (relative) of an FP32 rounding boundary, about 1 value
// in 10^7; such a value then differs by one FP32 ulp.
//
//  f64_log(x), x > 0 finite and normal:
//    x = 2^e * m with m in [sqrt(1/2), sqrt(2)), f = m - 1 (exact), and
//    log(m) = 2 atanh(s), s = f / (2 + f), |s| <= 0.1716.  With hfsq = f^2 / 2
//    one has 2s = f - hfsq + s * hfsq, so
//      log(m) = f - hfsq + s * (hfsq + R),   R = sum_{n>=1} 2 s^(2n) / (2n+1)
//    (the arrangement of Sun's fdlibm e_log.c; the coefficients here are the
//    series' own 2 / (2n+1), n = 1..11: the first term left out is below
//    2^-60 of the result).  e * ln2 is added as e * ln2_hi (exact product:
//    ln2_hi has 11 trailing zero bits) plus e * ln2_lo.
//  f64_exp(y), |y| < 700:
//    y = n * ln2 + r, n = rint(y / ln2), r reduced with the same split of
//    ln2 (|r| <= 0.347), exp(r) = sum_{k=0}^{13} r^k / k! by Horner
//    (remainder below 4e-18), scaled by 2^n.
//  f64_pow(t, c) = f64_exp(c * f64_log(t)), t > 0: the logarithm's absolute
//    error (a few 1e-17 for the |log t| < 3 of the callers) times c stays
//    far below an FP64 ulp of the product.
//  f64_pow_full(t, c), t > 0 finite and normal: the same series, with the terms
//    that carry more than 1/100 ulp of the result as unevaluated sums of two
//    doubles (Dekker's and Knuth's error-free sums and products, by FMA): s, s^3
//    / 3 and e ln2 of the logarithm, its product with c, and 1 + r + r^2 / 2 +
//    r^3 / 6 of the exponential (whose series goes to r^14 here).  Within 0.507
//    ulp of t^c: the final rounding, 0.001 for the logarithm's plain terms (2^-64
//    of its value, for |c log t| < 2), 0.001 for the first term left out
//    (0.347^15 / 15!) and 0.005 for the plain terms from r^4 / 24 on.
//  f64_div_by(x, c, rc), rc = RN(1 / c): x / c rounded once, as the IEEE
//    division rounds it (Markstein: the quotient x rc is within an ulp, its
//    remainder by FMA is exact and the corrected quotient rounds correctly, for
//    results in the normal range); zeros, infinities and NaN give what x / c gives
//    (the remainder is NaN there, and the quotient stands).
//
// Only FMA-explicit arithmetic (__builtin_fma) and IEEE operations, so the
// host and the device evaluate it to the same bits; tests/test_f64math.py
// compiles this header for the host and compares the FP32-rounded results
// with the C library's log and pow over every FP32 input of the callers'
// ranges.
#pragma once

#ifdef __HIPCC__
#define F64M_FN __host__ __device__ __forceinline__
#else
#define F64M_FN static inline
#endif

// ln 2 = kLn2Hi + kLn2Lo; kLn2Hi has its low 11 bits zero
#define F64M_LN2_HI 6.93147180369123816490e-01
#define F64M_LN2_LO 1.90821492927058770002e-10

F64M_FN double f64_log(double x) {
  int e;
  double m = __builtin_frexp(x, &e);  // [0.5, 1)
  if (m < 0.70710678118654752440) {
    m = m + m;
    e = e - 1;
  }
  const double f = m - 1.0;
  const double s = f / (2.0 + f);
  const double z = s * s;
  // R = z * (2/3 + z * (2/5 + ... + z * 2/23))
  double p = 2.0 / 23.0;
  p = __builtin_fma(p, z, 2.0 / 21.0);
  p = __builtin_fma(p, z, 2.0 / 19.0);
  p = __builtin_fma(p, z, 2.0 / 17.0);
  p = __builtin_fma(p, z, 2.0 / 15.0);
  p = __builtin_fma(p, z, 2.0 / 13.0);
  p = __builtin_fma(p, z, 2.0 / 11.0);
  p = __builtin_fma(p, z, 2.0 / 9.0);
  p = __builtin_fma(p, z, 2.0 / 7.0);
  p = __builtin_fma(p, z, 2.0 / 5.0);
  p = __builtin_fma(p, z, 2.0 / 3.0);
  const double R = z * p;
  const double hfsq = 0.5 * f * f;
  const double de = (double)e;
  // e*ln2_hi + (f - (hfsq - (s*(hfsq + R) + e*ln2_lo)))
  const double corr = __builtin_fma(s, hfsq + R, de * F64M_LN2_LO);
  return de * F64M_LN2_HI + (f - (hfsq - corr));
}

F64M_FN double f64_exp(double y) {
  const double n = __builtin_rint(y * 1.44269504088896338700);  // y / ln2
  const double r = __builtin_fma(-n, F64M_LN2_LO, __builtin_fma(-n, F64M_LN2_HI, y));
  // sum_{k=0}^{13} r^k / k!
  double p = 1.0 / 6227020800.0;  // 1/13!
  p = __builtin_fma(p, r, 1.0 / 479001600.0);
  p = __builtin_fma(p, r, 1.0 / 39916800.0);
  p = __builtin_fma(p, r, 1.0 / 3628800.0);
  p = __builtin_fma(p, r, 1.0 / 362880.0);
  p = __builtin_fma(p, r, 1.0 / 40320.0);
  p = __builtin_fma(p, r, 1.0 / 5040.0);
  p = __builtin_fma(p, r, 1.0 / 720.0);
  p = __builtin_fma(p, r, 1.0 / 120.0);
  p = __builtin_fma(p, r, 1.0 / 24.0);
  p = __builtin_fma(p, r, 1.0 / 6.0);
  p = __builtin_fma(p, r, 0.5);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_ldexp(p, (int)n);
}

F64M_FN double f64_pow(double t, double c) { return f64_exp(c * f64_log(t)); }

F64M_FN double f64_pow_full(double t, double c) {
  int e;
  double m = __builtin_frexp(t, &e);
  if (m < 0.70710678118654752440) {
    m = m + m;
    e = e - 1;
  }
  // s + sl = f / (2 + f), z + zl = s^2, q + ql = s^3
  const double f = m - 1.0, d = 2.0 + f, dl = f - (d - 2.0);
  const double rd = 1.0 / d, s = f * rd, sl = (__builtin_fma(-s, d, f) - s * dl) * rd;
  const double z = s * s, zl = __builtin_fma(s, s, -z) + 2.0 * s * sl;
  const double q = s * z, ql = __builtin_fma(s, z, -q) + (s * zl + sl * z);
  // h + l = log(m) / 2 = s + s^3 / 3 + s^5 (1/5 + s^2 / 7 + ... + s^18 / 23)
  const double c3 = 1.0 / 3.0, c3l = c3 / 18014398509481984.0;  // 1/3 in two parts: RN(1/3) = (1 - 2^-54) / 3
  const double w = q * c3, wl = __builtin_fma(q, c3, -w) + (q * c3l + ql * c3);
  double p = 1.0 / 23.0;
  p = __builtin_fma(p, z, 1.0 / 21.0);
  p = __builtin_fma(p, z, 1.0 / 19.0);
  p = __builtin_fma(p, z, 1.0 / 17.0);
  p = __builtin_fma(p, z, 1.0 / 15.0);
  p = __builtin_fma(p, z, 1.0 / 13.0);
  p = __builtin_fma(p, z, 1.0 / 11.0);
  p = __builtin_fma(p, z, 1.0 / 9.0);
  p = __builtin_fma(p, z, 1.0 / 7.0);
  p = __builtin_fma(p, z, 1.0 / 5.0);
  const double hi = s + w, lo = (w - (hi - s)) + ((sl + wl) + q * z * p);
  const double h = hi + lo, l = lo - (h - hi);
  // y + yl = c (e ln2 + log(m))
  const double de = (double)e, A = de * F64M_LN2_HI, L = A + 2.0 * h;
  const double Ll = (2.0 * h - (L - A)) + __builtin_fma(de, F64M_LN2_LO, 2.0 * l);
  const double y = c * L, yl = __builtin_fma(c, L, -y) + c * Ll;
  // r + rl = y - n ln2
  const double n = __builtin_rint(y * 1.44269504088896338700);
  const double r0 = __builtin_fma(-n, F64M_LN2_HI, y), r1 = __builtin_fma(-n, F64M_LN2_LO, yl);
  const double r = r0 + r1, rl = r1 - (r - r0);
  // g + (the rest) = exp(r + rl)
  const double r2 = r * r, r2l = __builtin_fma(r, r, -r2);
  const double r3 = r * r2, r3l = __builtin_fma(r, r2, -r3) + r * r2l;
  const double c6 = 0.5 * c3, u = r3 * c6, ul = __builtin_fma(r3, c6, -u) + (r3 * (0.5 * c3l) + r3l * c6);
  double v = 1.0 / 87178291200.0;  // 1/14!
  v = __builtin_fma(v, r, 1.0 / 6227020800.0);
  v = __builtin_fma(v, r, 1.0 / 479001600.0);
  v = __builtin_fma(v, r, 1.0 / 39916800.0);
  v = __builtin_fma(v, r, 1.0 / 3628800.0);
  v = __builtin_fma(v, r, 1.0 / 362880.0);
  v = __builtin_fma(v, r, 1.0 / 40320.0);
  v = __builtin_fma(v, r, 1.0 / 5040.0);
  v = __builtin_fma(v, r, 1.0 / 720.0);
  v = __builtin_fma(v, r, 1.0 / 120.0);
  v = __builtin_fma(v, r, 1.0 / 24.0);
  const double a = 1.0 + r, b = a + 0.5 * r2, g = b + u;
  const double rest = ((u - (g - b)) + ((0.5 * r2 - (b - a)) + (r - (a - 1.0)))) + (r2 * r2 * v + ((0.5 * r2l + ul) + rl * g));
  return __builtin_ldexp(g + rest, (int)n);
}

F64M_FN double f64_div_by(double x, double c, double rc) {
  const double q = x * rc, v = __builtin_fma(__builtin_fma(-q, c, x), rc, q);
  return v == v ? v : q;
}
