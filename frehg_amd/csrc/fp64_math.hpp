// FP64 log, exp, expm1 and log1p for the van Genuchten relations: in well under half of the instructions of
// the general library functions, and with arguments and logarithms as unevaluated sums of two doubles, so that
// powers x^a = exp(a log x) and differences of logarithms lose nothing between the two steps. The Richards
// kernels that evaluate the relations are bound by FP64 vector instructions (490 to 670 per wave with the
// library functions, DRAM idle), so the instruction count is their time.
//
// Methods (textbook argument reduction and error-free transformations; the polynomials are fitted for this file
// by Remez exchange in 50-digit arithmetic):
//   log     x = 2^e m, m in [sqrt(1/2), sqrt(2)); with s = (m - 1)/(m + 1), log m = 2 atanh s = 2s + s z R(z),
//           z = s^2; s = s0 + residual from a Newton reciprocal, with the rounding error of m + 1.
//   exp     k = round(x / ln 2), r = x - k ln 2 (|r| <= ln 2 / 2) as r + rl, 2^k (1 + r + rl + r^2 Q(r)).
//   expm1   the same r: 2^k (r + rl + r^2 Q(r)) + (2^k - 1).
//   log1p   log(u) + err / u with u + err = 1 + x exactly.
// Explicit fma and no contraction, so that every kernel gets the same bits for the same argument.
//
// Against 60-digit values exp and expm1 are within 0.8 units in the last place, the pairs within 2^-56.5 of the
// logarithm's size (x in [0.5, 2]; elsewhere 2^-58), that of log1p within 2^-53.5 for x below 1e-12. NaN gives NaN;
// exp and expm1 saturate through ldexp; the logarithms of 0, of negative numbers and of infinity are the
// caller's to exclude.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace frehg {
namespace fm {

struct Two {  // hi + lo, |lo| at most about an ulp of hi
  double hi, lo;
};

// 1/x by two Newton steps for x of moderate size: within an ulp.
__host__ __device__ __forceinline__ double recip(double x) {
#pragma clang fp contract(off)
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(x);
#else
  double y = (double)(1.0f / (float)x);  // (a coarser start than the device's; the steps converge either way)
#endif
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}

// a * (b.hi + b.lo).
__host__ __device__ __forceinline__ Two mul(double a, Two b) {
#pragma clang fp contract(off)
  const double h = a * b.hi;
  return Two{h, fma(a, b.lo, fma(a, b.hi, -h))};
}

// a + b for |a| >= |b|.
__host__ __device__ __forceinline__ Two add(Two a, double b) {
#pragma clang fp contract(off)
  const double h = a.hi + b;
  return Two{h, (b - (h - a.hi)) + a.lo};
}

// a - b.
__host__ __device__ __forceinline__ Two sub(Two a, Two b) {
#pragma clang fp contract(off)
  const double h = a.hi - b.hi, t = h - a.hi;
  return Two{h, ((a.hi - (h - t)) - (b.hi + t)) + (a.lo - b.lo)};
}

// (2 atanh(s) / s - 2) / z with z = s^2, |s| <= 0.1716.
__host__ __device__ __forceinline__ double atanh_tail(double z) {
#pragma clang fp contract(off)
  double R = 1.30885160094571740e-01;
  R = fma(R, z, 1.32685835548657288e-01);
  R = fma(R, z, 1.53862471690389829e-01);
  R = fma(R, z, 1.81817954944370724e-01);
  R = fma(R, z, 2.22222223931722418e-01);
  R = fma(R, z, 2.85714285707966698e-01);
  R = fma(R, z, 4.00000000000008904e-01);
  return fma(R, z, 6.66666666666666630e-01);
}

// log(x) + add, |add| small against the result's ulps' neighbourhood (the tail of log1p), x > 0 finite.
__host__ __device__ __forceinline__ Two log(double x, double add = 0.0) {
#pragma clang fp contract(off)
  int e;
  double m;
#if defined(__HIP_DEVICE_COMPILE__)
  m = __builtin_amdgcn_frexp_mant(x);
  e = __builtin_amdgcn_frexp_exp(x);
#else
  m = std::frexp(x, &e);
#endif
  const int low = m < 0.70710678118654757 ? 1 : 0;
  m = ldexp(m, low);
  const double k = (double)(e - low);
  const double n = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);  // d + dl = m + 1
  const double y = recip(d);
  const double s = n * y;
  const double sl = fma(-s, dl, fma(-s, d, n)) * y;  // n / (m + 1) = s + sl
  const double z = s * s;
  const double R = atanh_tail(z);
  const double c = k * 6.93147180369123816e-01;  // (exact: 32 bits times a small integer)
  const double h1 = fma(2.0, s, c);
  const double e1 = fma(2.0, s, c - h1);
  const double lo = fma(k, 1.90821492927058770e-10, fma(s, z * R, fma(2.0, sl, add))) + e1;
  const double h = h1 + lo;
  return Two{h, lo - (h - h1)};
}

// k, r and rl of exp and expm1: x = k ln 2 + r + rl.
__host__ __device__ __forceinline__ double reduce(Two x, double* r, double* rl) {
#pragma clang fp contract(off)
  const double kd = rint(x.hi * 1.44269504088896339e+00);
  const double r0 = fma(kd, -6.93147180369123816e-01, x.hi);
  *r = fma(kd, -1.90821492927058770e-10, r0);
  *rl = fma(kd, -1.90821492927058770e-10, r0 - *r) + x.lo;
  return kd;
}

__host__ __device__ __forceinline__ int exponent(double kd) { return (int)fmin(fmax(kd, -2200.0), 2200.0); }

// rl + expm1(r) - r.
__host__ __device__ __forceinline__ double expm1_tail(double r, double rl) {
#pragma clang fp contract(off)
  double q = 2.09216072466720266e-09;
  q = fma(q, r, 2.51052599225407319e-08);
  q = fma(q, r, 2.75572528671516270e-07);
  q = fma(q, r, 2.75572552971325119e-06);
  q = fma(q, r, 2.48015873473784143e-05);
  q = fma(q, r, 1.98412698749017926e-04);
  q = fma(q, r, 1.38888888888743850e-03);
  q = fma(q, r, 8.33333333332611156e-03);
  q = fma(q, r, 4.16666666666666852e-02);
  q = fma(q, r, 1.66666666666666713e-01);
  q = fma(q, r, 5.00000000000000000e-01);
  return fma(r * r, q, fma(rl, r, rl));
}

__host__ __device__ __forceinline__ double exp(Two x) {
#pragma clang fp contract(off)
  double r, rl;
  const double kd = reduce(x, &r, &rl);
  const double w = 1.0 + r;
  return ldexp(w + ((r - (w - 1.0)) + expm1_tail(r, rl)), exponent(kd));
}

__host__ __device__ __forceinline__ double expm1(Two x) {
#pragma clang fp contract(off)
  double r, rl;
  const double kd = reduce(x, &r, &rl);
  const double q = expm1_tail(r, rl);
  const int k = exponent(kd);
  const double t = ldexp(1.0, k), c = t - 1.0;
  const double h = fma(t, r, c);
  return k > 60 ? ldexp(1.0 + (r + q), k) : h + fma(t, q, fma(t, r, c - h));
}

// log(1 + x) for x >= 0.
__host__ __device__ __forceinline__ Two log1p(double x) {
#pragma clang fp contract(off)
  const double u = 1.0 + x, b = u - 1.0;
  const double err = (1.0 - (u - b)) + (x - b);
  return log(u, err * recip(u));
}

// log(1 + 1/x) for x >= 2.42: 2 atanh(1 / (2 x + 1)), to an ulp or two however small.
__host__ __device__ __forceinline__ double log1p_inverse(double x) {
#pragma clang fp contract(off)
  const double s = recip(fma(2.0, x, 1.0)), z = s * s;
  return fma(s, z * atanh_tail(z), 2.0 * s);
}

}  // namespace fm
}  // namespace frehg
