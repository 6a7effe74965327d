// pow(x, y) for finite x > 0 evaluated in double-double arithmetic (about
// 100 significant bits) and rounded once, so the result is the correctly
// rounded x^y except when x^y lies within ~2^-100 (relative) of a rounding
// boundary.  The step-size controller needs pow(err, 1/(1+q)) each attempt
// (RKEmbeddedParallel.hpp:24, :65, :198); a correctly rounded value is
// platform independent, so the device controller and any host controller
// choose identical step sizes.
//
// Method: x = 2^e m with m in [sqrt(1/2), sqrt(2)); log m = 2 atanh(u),
// u = (m-1)/(m+1), by its odd power series (|u| <= 0.1716, 22 terms);
// z = y log x; exp z = 2^k exp(r) with r = z - k ln2, exp(r) from the Taylor
// series of exp(r/256) - 1 followed by eight squarings in the expm1 form
// s <- 2s + s^2.  Only +, -, *, fma and exact scaling are used, so the host
// and device builds produce the same bits.  Callers must compile with FMA
// contraction off (explicit fma is still fused).
#pragma once

#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#define ODEHIP_HD __host__ __device__
#else
#define ODEHIP_HD
#endif

namespace odehip {
namespace crpow_detail {

struct dd {
  double hi, lo;
};

ODEHIP_HD inline uint64_t to_bits(double x) { return __builtin_bit_cast(uint64_t, x); }
ODEHIP_HD inline double from_bits(uint64_t b) { return __builtin_bit_cast(double, b); }

ODEHIP_HD inline dd two_sum(double a, double b) {
  double s = a + b;
  double bb = s - a;
  double e = (a - (s - bb)) + (b - bb);
  return {s, e};
}
ODEHIP_HD inline dd quick_two_sum(double a, double b) {
  double s = a + b;
  double e = b - (s - a);
  return {s, e};
}
ODEHIP_HD inline dd two_prod(double a, double b) {
  double p = a * b;
  double e = std::fma(a, b, -p);
  return {p, e};
}
ODEHIP_HD inline dd add(dd a, dd b) {
  dd s = two_sum(a.hi, b.hi);
  dd t = two_sum(a.lo, b.lo);
  s.lo += t.hi;
  s = quick_two_sum(s.hi, s.lo);
  s.lo += t.lo;
  return quick_two_sum(s.hi, s.lo);
}
ODEHIP_HD inline dd mul(dd a, dd b) {
  dd p = two_prod(a.hi, b.hi);
  p.lo += a.hi * b.lo + a.lo * b.hi;
  return quick_two_sum(p.hi, p.lo);
}
ODEHIP_HD inline dd mul_d(dd a, double b) {
  dd p = two_prod(a.hi, b);
  p.lo += a.lo * b;
  return quick_two_sum(p.hi, p.lo);
}
ODEHIP_HD inline dd div(dd a, dd b) {
  double q1 = a.hi / b.hi;
  dd r = add(a, mul_d(b, -q1));
  double q2 = r.hi / b.hi;
  r = add(r, mul_d(b, -q2));
  double q3 = r.hi / b.hi;
  dd q = quick_two_sum(q1, q2);
  return add(q, dd{q3, 0.0});
}
// Exact power-of-two scaling through the exponent field.
ODEHIP_HD inline double scale2(double v, int k) {
  // k is small (|k| < 1000 here); split to stay in the normal range.
  while (k > 1000) {
    v *= 0x1p1000;
    k -= 1000;
  }
  while (k < -1000) {
    v *= 0x1p-1000;
    k += 1000;
  }
  return v * from_bits(static_cast<uint64_t>(k + 1023) << 52);
}

// 1 / (2k + 1), k = 0 .. 21, and 1 / k!, k = 0 .. 11, to double-double: 66
// divisions a call were half of its time on the controller's one lane.
constexpr dd kOddInverse[22] = {
    {0x1.0000000000000p+0, 0x0.0p+0},
    {0x1.5555555555555p-2, 0x1.5555555555555p-56},
    {0x1.999999999999ap-3, -0x1.999999999999ap-57},
    {0x1.2492492492492p-3, 0x1.2492492492492p-57},
    {0x1.c71c71c71c71cp-4, 0x1.c71c71c71c71cp-58},
    {0x1.745d1745d1746p-4, -0x1.745d1745d1746p-59},
    {0x1.3b13b13b13b14p-4, -0x1.3b13b13b13b14p-58},
    {0x1.1111111111111p-4, 0x1.1111111111111p-60},
    {0x1.e1e1e1e1e1e1ep-5, 0x1.e1e1e1e1e1e1ep-61},
    {0x1.af286bca1af28p-5, 0x1.af286bca1af28p-59},
    {0x1.8618618618618p-5, 0x1.8618618618618p-59},
    {0x1.642c8590b2164p-5, 0x1.642c8590b2164p-60},
    {0x1.47ae147ae147bp-5, -0x1.eb851eb851eb8p-61},
    {0x1.2f684bda12f68p-5, 0x1.2f684bda12f68p-59},
    {0x1.1a7b9611a7b96p-5, 0x1.1a7b9611a7b96p-61},
    {0x1.0842108421084p-5, 0x1.0842108421084p-60},
    {0x1.f07c1f07c1f08p-6, -0x1.f07c1f07c1f08p-61},
    {0x1.d41d41d41d41dp-6, 0x1.0750750750750p-60},
    {0x1.bacf914c1bad0p-6, -0x1.bacf914c1bad0p-60},
    {0x1.a41a41a41a41ap-6, 0x1.0690690690690p-60},
    {0x1.8f9c18f9c18fap-6, -0x1.f3831f3831f38p-61},
    {0x1.7d05f417d05f4p-6, 0x1.7d05f417d05f4p-62},
};
constexpr dd kInverseFactorial[12] = {
    {0x1.0000000000000p+0, 0x0.0p+0},
    {0x1.0000000000000p+0, 0x0.0p+0},
    {0x1.0000000000000p-1, 0x0.0p+0},
    {0x1.5555555555555p-3, 0x1.5555555555555p-57},
    {0x1.5555555555555p-5, 0x1.5555555555555p-59},
    {0x1.1111111111111p-7, 0x1.1111111111111p-63},
    {0x1.6c16c16c16c17p-10, -0x1.f49f49f49f49fp-65},
    {0x1.a01a01a01a01ap-13, 0x1.a01a01a01a01ap-73},
    {0x1.a01a01a01a01ap-16, 0x1.a01a01a01a01ap-76},
    {0x1.71de3a556c734p-19, -0x1.c154f8ddc6c00p-73},
    {0x1.27e4fb7789f5cp-22, 0x1.cbbc05b4fa99ap-76},
    {0x1.ae64567f544e4p-26, -0x1.c062e06d1f209p-80},
};

// ln 2 to ~107 bits.
constexpr double kLn2Hi = 6.93147180559945286227e-01;
constexpr double kLn2Lo = 2.31904681384629955842e-17;

ODEHIP_HD inline dd log_dd(double x) {
  // x finite, > 0, normal.
  const uint64_t bits = to_bits(x);
  int e = static_cast<int>((bits >> 52) & 0x7ff) - 1023;
  uint64_t mbits = (bits & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL;
  double m = from_bits(mbits);  // m in [1, 2)
  if (m > 1.4142135623730951) {
    m *= 0.5;
    e += 1;
  }
  // u = (m - 1) / (m + 1); m - 1 is exact (Sterbenz), m + 1 as double-double.
  dd num{m - 1.0, 0.0};
  dd den = two_sum(m, 1.0);
  dd u = div(num, den);
  dd w = mul(u, u);
  // sum_{k=0}^{21} w^k / (2k+1), Horner from the top.
  dd s = kOddInverse[21];
#pragma unroll
  for (int k = 20; k >= 0; --k) {
    s = add(mul(s, w), kOddInverse[k]);
  }
  dd lm = mul(mul_d(u, 2.0), s);
  dd le = add(two_prod(static_cast<double>(e), kLn2Hi),
              dd{static_cast<double>(e) * kLn2Lo, 0.0});
  return add(le, lm);
}

ODEHIP_HD inline double exp_dd_round(dd z) {
  double kd = std::nearbyint(z.hi / kLn2Hi);
  int k = static_cast<int>(kd);
  // r = z - k ln2
  dd kl = add(two_prod(kd, kLn2Hi), two_prod(kd, kLn2Lo));
  dd r = add(z, dd{-kl.hi, -kl.lo});
  // r' = r / 256 (exact)
  dd rp{r.hi * 0.00390625, r.lo * 0.00390625};
  // s = exp(r') - 1 = r' + r'^2/2! + ... + r'^11/11!
  dd s = kInverseFactorial[11];
#pragma unroll
  for (int n = 10; n >= 1; --n) {
    s = add(mul(s, rp), kInverseFactorial[n]);
  }
  s = mul(s, rp);
  for (int i = 0; i < 8; ++i) {
    // (1 + s)^2 - 1 = 2 s + s^2
    s = add(dd{2.0 * s.hi, 2.0 * s.lo}, mul(s, s));
  }
  dd v = add(dd{1.0, 0.0}, s);
  double hi = v.hi + v.lo;  // round the double-double once
  return scale2(hi, k);
}

}  // namespace crpow_detail

// Correctly rounded (see above) x^y for x > 0 finite normal, y finite, and a
// result in the normal range.  pow(0, y>0) = 0; other special inputs fall back
// to the IEEE conventions of the C library's pow.
ODEHIP_HD inline double cr_pow(double x, double y) {
  using namespace crpow_detail;
  if (x == 1.0 || y == 0.0) return 1.0;
  if (!(x > 0.0) || !std::isfinite(x) || !std::isfinite(y) ||
      x < 2.2250738585072014e-308) {
    return std::pow(x, y);
  }
  dd l = log_dd(x);
  dd z = mul_d(l, y);
  if (z.hi > 709.0 || z.hi < -708.0) return std::pow(x, y);
  return exp_dd_round(z);
}

// x^y for y = the double nearest to 1 / k, k an integer >= 2: the same value as
// cr_pow(x, y) (correctly rounded but within ~2^-98 of a tie), by a shorter way
// than logarithm and exponential: the controller runs on one lane while
// everything else waits, and cr_pow's two series take it 7 us of dependent
// arithmetic on MI355X, this about 1.
//
// r, a k-th root of x to a few ulp, comes from FP32 log2 / exp2 and Newton
// steps.  With P = r^k in double-double and s = (x - P) / x (P.hi and x are
// neighbours, so the difference is exact), x^(1/k) = r (1 - s)^(-1/k), and
// x^y = x^(1/k) x^d with d = y - 1/k known exactly from the fma residual, so x^y is
// r (1 + s/k + (1/k + 1) s^2 / (2 k)) (1 + z + z^2/2), z = d log x: one rounding
// of r plus a correction of some 2^-51 r.
ODEHIP_HD inline double cr_root(double x, double y, int k) {
  using namespace crpow_detail;
  if (!(x >= 0x1p-900 && x <= 0x1p900) || k < 2 || k > 64) return cr_pow(x, y);
  if (x == 1.0) return 1.0;
  const uint64_t bits = to_bits(x);
  const int e = static_cast<int>(bits >> 52) - 1023;
  const double m = from_bits((bits & 0x000fffffffffffffULL) | 0x3ff0000000000000ULL);
  const double ix = 1.0 / x;
  const double d = std::fma(y, static_cast<double>(k), -1.0) * y;  // y - 1/k
  const double z = d != 0.0 ? d * std::log(x) : 0.0;
  const double l = (static_cast<double>(e) + static_cast<double>(log2f(static_cast<float>(m)))) * y;
  const double n = std::nearbyint(l);
  double r = static_cast<double>(exp2f(static_cast<float>(l - n))) *
             from_bits(static_cast<uint64_t>(static_cast<int>(n) + 1023) << 52);
  for (int it = 0; it < 2; ++it) {  // 1e-6 -> 1e-11 -> rounding
    double p = r;
    for (int i = 1; i < k; ++i) p *= r;
    r += r * (((x - p) * ix) * y);
  }
  dd p{r, 0.0};
  for (int i = 1; i < k; ++i) p = mul_d(p, r);
  const double s = ((x - p.hi) - p.lo) * ix;
  const double c = (s * y) * (1.0 + s * (0.5 * y + 0.5));
  const double w = z + 0.5 * z * z;
  return r + r * (c + w + c * w);
}

}  // namespace odehip
