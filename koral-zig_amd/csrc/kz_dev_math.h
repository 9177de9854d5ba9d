// kz_dev_math.h — the transcendentals of kz_math.h for gfx950, without
// branches: every result equals kz_math.h's bit for bit (NaN for NaN).
//
// A branch ends the block that the compiler schedules, so kz_math.h's early
// returns keep two functions of independent operands from overlapping, and a
// wave that has its SIMD to itself (the implicit kernels) then waits out each
// FP64 latency in turn: the radiation residual with its log1p, three powers of
// one base each, two cube roots and two exponentials took 11 500 cycles for
// about 2000 instructions.  Here special operands are selected at the end,
// the exponent field is taken and set by v_frexp / v_ldexp (which also treat
// subnormals, with the one rounding that kz_math.h's two-step scaling makes),
// and products that kz_math.h notes as exact are fused.
//
//   kzm_exp_dd     x > 709.78 is +inf, x < -745.13 is 0; NaN passes through
//   kzm_log        0 gives -inf, +inf itself, negative and NaN give NaN
//   kzm_pow        a finite positive exponent that is no integer, from the
//                  base's logarithm (shared by several powers of one base)
#pragma once

#include "kz_math.h"

#define KZDM __device__ static __forceinline__

namespace kzd {

KZDM double dm_sel(bool c, double a, double b) { return c ? a : b; }

// x toward zero as an integer for every x: past the range the nearest value in
// it, 0 for NaN, which is what the instruction gives.  A cast is undefined for
// those operands (dm_exp_dd selects its result only afterwards), and what keeps
// them from one costs.  Implicit pass at 384x360 and 128x128x32: a bare cast 290
// and 842 us, this 288 and 819, x clamped before a cast 290 and 881, clamped in
// FP32 295 and 846; the low word of x + 1.5 * 2^52 made 40 whole steps at
// 128x128x32 2.3 % slower.
KZDM int dm_int(double x) {
  int k;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(x));
  return k;
}

// kzm_exp_dd
KZDM double dm_exp_dd(double x, double xl) {
  const double t = x * KZM_INV_LN2;
  const double kd = __builtin_trunc(t + __builtin_copysign(0.5, t));
  const double hi = KZM_FMA(-kd, KZM_LN2_HI, x);  // the product is exact
  const double lo = KZM_FMA(kd, KZM_LN2_LO, -xl);
  const double r = hi - lo;
  const double c = (hi - r) - lo;
  double q = 0x1.6124613a86d09p-33;
  q = KZM_FMA(r, q, 0x1.1eed8eff8d898p-29);
  q = KZM_FMA(r, q, 0x1.ae64567f544e4p-26);
  q = KZM_FMA(r, q, 0x1.27e4fb7789f5cp-22);
  q = KZM_FMA(r, q, 0x1.71de3a556c734p-19);
  q = KZM_FMA(r, q, 0x1.a01a01a01a01ap-16);
  q = KZM_FMA(r, q, 0x1.a01a01a01a01ap-13);
  q = KZM_FMA(r, q, 0x1.6c16c16c16c17p-10);
  q = KZM_FMA(r, q, 0x1.1111111111111p-7);
  q = KZM_FMA(r, q, 0x1.5555555555555p-5);
  q = KZM_FMA(r, q, 0x1.5555555555555p-3);
  q = KZM_FMA(r, q, 0.5);
  q = (r * r) * q;
  const double y = 1.0 + (r + (q + c * (1.0 + r)));
  const double v = __builtin_amdgcn_ldexp(y, dm_int(kd));
  return dm_sel(x > 709.782712893384, KZM_INF, dm_sel(x < -745.1332191019412, 0.0, v));
}
KZDM double dm_exp(double x) { return dm_exp_dd(x, 0.0); }

// kzm_log_dd (finite x > 0; anything else gives a value to be selected away)
KZDM void dm_log_dd(double x, double *hi_out, double *lo_out) {
  const double fm = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
  const int fe = __builtin_amdgcn_frexp_exp(x);
  const bool up = fm > 0x1.6a09e667f3bcdp-1;  // above sqrt(1/2): m = fm, else m = 2 fm
  const double m = dm_sel(up, fm, fm + fm);
  const double ed = (double)(up ? fe : fe - 1);
  const double f = m - 1.0;
  double uh, ul;
  kzm_fast_two_sum(2.0, f, &uh, &ul);
  const double inv = 1.0 / uh;
  const double sh = f * inv;
  const double sl = (KZM_FMA(-sh, uh, f) - sh * ul) * inv;
  const double s2 = sh * sh;
  double p = 0x1.642c8590b2164p-4;
  p = KZM_FMA(s2, p, 0x1.8618618618618p-4);
  p = KZM_FMA(s2, p, 0x1.af286bca1af28p-4);
  p = KZM_FMA(s2, p, 0x1.e1e1e1e1e1e1ep-4);
  p = KZM_FMA(s2, p, 0x1.1111111111111p-3);
  p = KZM_FMA(s2, p, 0x1.3b13b13b13b14p-3);
  p = KZM_FMA(s2, p, 0x1.745d1745d1746p-3);
  p = KZM_FMA(s2, p, 0x1.c71c71c71c71cp-3);
  p = KZM_FMA(s2, p, 0x1.2492492492492p-2);
  p = KZM_FMA(s2, p, 0x1.999999999999ap-2);
  p = KZM_FMA(s2, p, 0x1.5555555555555p-1);
  const double tail = (s2 * sh) * p;
  const double a = ed * KZM_LN2_HI;
  double hi, err;
  kzm_two_sum(a, 2.0 * sh, &hi, &err);
  const double lo = err + (ed * KZM_LN2_LO + (2.0 * sl + tail));
  kzm_fast_two_sum(hi, lo, hi_out, lo_out);
}
// kzm_log
KZDM double dm_log(double x) {
  double h, l;
  dm_log_dd(x, &h, &l);
  h = dm_sel(x > 0.0, h, dm_sel(x == 0.0, -KZM_INF, KZM_NAN));
  return dm_sel(x == KZM_INF, KZM_INF, h);
}
// kzm_pow_from_log for y != 0
KZDM double dm_pow_from_log(double lh, double ll, double y) {
  double zh, zl, th, tl;
  kzm_two_prod(y, lh, &zh, &zl);
  zl += y * ll;
  kzm_fast_two_sum(zh, zl, &th, &tl);
  return dm_exp_dd(th, tl);
}
// kzm_pow(x, y) for a finite y > 0 that is no integer, `raw` being
// dm_pow_from_log of x's logarithm
KZDM double dm_pow_fix(double x, double raw) {
  const double r = dm_sel(x > 0.0, raw, dm_sel(x == 0.0, 0.0, KZM_NAN));
  return dm_sel(x == KZM_INF, KZM_INF, r);
}
KZDM double dm_pow_frac(double x, double y) {
  double h, l;
  dm_log_dd(x, &h, &l);
  return dm_pow_fix(x, dm_pow_from_log(h, l, y));
}
// kzm_cbrt
KZDM double dm_cbrt(double x) {
  const double ax = kzm_fabs(x);
  const int et = __builtin_amdgcn_frexp_exp(ax) - 1;
  // floor(et / 3) for -1100 < et < 1100
  const int j = (int)(((unsigned)(et + 3072) * 43691u) >> 17) - 1024;
  const int r3 = et - 3 * j;
  const double m =
      kzm_from_bits((kzm_bits(__builtin_amdgcn_frexp_mant(ax)) & 0x000fffffffffffffULL) | ((uint64_t)(1023 + r3) << 52));
  double y = kzm_from_bits(0x5540000000000000ULL - kzm_bits(m) / 3);
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const double y3 = (y * y) * y;
    y = KZM_FMA(y * KZM_FMA(-m, y3, 1.0), 0x1.5555555555555p-2, y);
  }
  const double y2 = y * y;
  double t = m * y2;
  double p2h, p2l, p3h, p3l;
  kzm_two_prod(t, t, &p2h, &p2l);
  kzm_two_prod(p2h, t, &p3h, &p3l);
  p3l += p2l * t;
  const double resid = (m - p3h) - p3l;
  t = KZM_FMA(resid, y2 * 0x1.5555555555555p-2, t);
  const double v = __builtin_copysign(__builtin_amdgcn_ldexp(t, j), x);
  return dm_sel(ax > 0.0 && ax < KZM_INF, v, x);
}
// kzm_log1p
KZDM double dm_log1p(double x) {
  const double u = 1.0 + x;
  const double v = dm_sel(x < -1.0, KZM_NAN, dm_log(u) * (x / (u - 1.0)));
  return dm_sel(x == KZM_INF, KZM_INF, dm_sel(u == 1.0, x, v));
}
// log(p^(1/(gam-1)) / rho^(1/(gam-1) + 1)), the logarithm of the entropy
// function (hydro.zig:32-37, invert.zig:188): for positive finite p and rho
// the two powers run side by side, anything else takes kz_math.h's way
KZDM double dm_log_entropy(double p, double rho, double indexn) {
  if (p > 0.0 && p < KZM_INF && rho > 0.0 && rho < KZM_INF && kzm_isfinite(indexn) && indexn != 0.0 &&
      indexn != -1.0) {
    double ph, pl, rh, rl;
    dm_log_dd(p, &ph, &pl);
    dm_log_dd(rho, &rh, &rl);
    return dm_log(dm_pow_from_log(ph, pl, indexn) / dm_pow_from_log(rh, rl, indexn + 1.0));
  }
  // a negative pressure, as the trials of a damped W iteration meet it, has no
  // power: NaN without the rest
  if (p < 0.0 && kzm_isfinite(indexn) && __builtin_trunc(indexn) != indexn) return KZM_NAN;
  return kzm_log(kzm_pow(p, indexn) / kzm_pow(rho, indexn + 1.0));
}

}  // namespace kzd
