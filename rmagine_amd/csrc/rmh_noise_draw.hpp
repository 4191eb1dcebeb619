// Radius of the Box-Muller draw: sqrt(-2 log u) for u = m 2^-24, m = 1 .. 2^24, in FP64.  Shared
// by the noise kernels and their host check (tests/cpp/noise_radius_check.cpp, all 2^24 draws).
//
// log u: m = 2^e z with z in [0.707, 1.414] (integer operations on m as an FP32 value, which
// holds it exactly); s = (z - 1) / (z + 1), both exact; log z = 2 artanh s by its series to
// s^21 (|s| <= 0.1716: the next term is below 2e-18 of the first).  The low parts of the quotient
// and of e log 2 + 2 s are carried, so that log u is rounded once, and the root once: the largest
// relative error of all draws is 1.66e-16, the general functions' 1.68e-16 on the MI355X (without
// the low parts 2.14e-16, and 32.8M relative Gaussian ranges in 148 us instead of 155).  The
// general log and sqrt scale their arguments and order their special cases; with neither, about
// 60 FP64 instructions become 40.
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define RMH_DRAW_HD __host__ __device__ inline
#else
#define RMH_DRAW_HD inline
#endif

namespace rmh {

// x, its quotient, reciprocal and reciprocal root to about FP32 precision
#if defined(__HIP_DEVICE_COMPILE__)
RMH_DRAW_HD double rough_rcp(double x) { return __builtin_amdgcn_rcp(x); }
RMH_DRAW_HD double rough_rsq(double x) { return __builtin_amdgcn_rsq(x); }
// a b + k with the constant k from scalar registers: the compiler's form adds into the
// constant's copy in vector registers, two moves per coefficient
RMH_DRAW_HD double fma_const(double a, double b, double k) {
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(k));
  return r;
}
#else
#ifndef RMH_DRAW_ROUGH
#define RMH_DRAW_ROUGH 1.0
#endif
RMH_DRAW_HD double rough_rcp(double x) { return static_cast<double>(static_cast<float>(RMH_DRAW_ROUGH / x)); }
RMH_DRAW_HD double rough_rsq(double x) { return static_cast<double>(static_cast<float>(RMH_DRAW_ROUGH / std::sqrt(x))); }
RMH_DRAW_HD double fma_const(double a, double b, double k) { return std::fma(a, b, k); }
#endif

RMH_DRAW_HD double normal_radius(uint32_t m) {
  const float mf = static_cast<float>(m);
  uint32_t bits;
  std::memcpy(&bits, &mf, 4);
  // exponent such that z lies in [0.707, 1.414]: 0x3504F3 is sqrt 2's significand
  const uint32_t b = bits - 0x3F3504F3u;
  const int e = static_cast<int>(b >> 23) - 24;
  const uint32_t zb = (b & 0x7FFFFFu) + 0x3F3504F3u;
  float zf;
  std::memcpy(&zf, &zb, 4);
  const double z = static_cast<double>(zf);
  const double num = z - 1.0, den = z + 1.0;
  double y = rough_rcp(den);
  y = std::fma(std::fma(-den, y, 1.0), y, y);
  double s = num * y;
  s = std::fma(std::fma(-den, s, num), y, s);
  const double sl = std::fma(-den, s, num) * y;  // what s misses of the quotient
  const double w = s * s;
  double p = 2.0 / 21.0;
  p = fma_const(p, w, 2.0 / 19.0);
  p = fma_const(p, w, 2.0 / 17.0);
  p = fma_const(p, w, 2.0 / 15.0);
  p = fma_const(p, w, 2.0 / 13.0);
  p = fma_const(p, w, 2.0 / 11.0);
  p = fma_const(p, w, 2.0 / 9.0);
  p = fma_const(p, w, 2.0 / 7.0);
  p = fma_const(p, w, 2.0 / 5.0);
  p = fma_const(p, w, 2.0 / 3.0);
  // x = -2 log u >= 0; e ln 2 + 2 s is split into its rounded value and the rest (log 2's upper
  // part has 33 bits, so its product with e is exact), to which the small terms are added
  const double ed = static_cast<double>(e), s2 = s + s;
  const double t = std::fma(ed, 0x1.62e42fefp-1, s2);
  const double rest = std::fma(ed, 0x1.62e42fefp-1, -t) + s2;
  const double low = std::fma(ed, 0x1.473de6af278edp-34, std::fma(s * w, p, sl + sl) + rest);
  const double x = -2.0 * (t + low);
  // sqrt x by coupled Newton steps on g ~ sqrt x and h ~ 1 / (2 sqrt x)
  const double r = rough_rsq(x);
  double g = x * r, h = 0.5 * r;
  const double d = std::fma(-h, g, 0.5);
  g = std::fma(g, d, g);
  h = std::fma(h, d, h);
  g = std::fma(std::fma(-g, g, x), h, g);
  return m == 0x1000000u ? 0.0 : g;  // u = 1: x = 0, whose reciprocal root is infinite
}

}  // namespace rmh
