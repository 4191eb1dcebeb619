// Per-ray set-up of the FP32 slab test of the ray kernels (rmh_trace.hpp: slab2), compiled for
// the device and by its host check (tests/cpp/slab_length_check.cpp).
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define RMH_SLAB_HD __host__ __device__ __forceinline__
#else
#define RMH_SLAB_HD inline
#endif

#ifndef RMH_SLAB_RECIPROCAL  // the check puts other reciprocals in
#define RMH_SLAB_RECIPROCAL(x) (1.0f / (x))
#endif

namespace rmh {

// Slab test.  A slab value is fma(plane, 1/d, -(o +- P) / d) with a per-ray margin
//   P = 2^-21 (max|o| + range_max) + 1e-30.
// Written out, a computed value is t' = (plane - o -+ P'') / d * (1 + r), where
//   * P'' lies in [0.74 P, 1.26 P]: o +- P and its product with 1/d are rounded, at most
//     2^-23 (|o| + P) <= P / 4 in position (the lo plane takes o + P, the hi plane o - P,
//     so both planes move outward);
//   * |r| <= 1.2e-7: the roundings of the exact division 1/d and of the fma.  (With the
//     reciprocal instruction, 1 ulp in one instruction instead of ten, |r| reaches 1.8e-7; it
//     saved 0.2 to 0.5 % of a cast, 8,669 -> 8,649 us for 1,000 scans of 128 x 1,024.)
// Replacing a direction component below 2^-64 by +-2^-64 moves the ray by at most
// range_max 2^-64, far below P.  Let the exact ray meet the box at some t <= range_max in
// [0, tbf] (tbf: an FP32 bound at least the closest hit found so far).  On each axis the near
// plane's exact crossing is <= t, so its moved plane crosses at <= t - P''/|d| and the computed
// near value is <= t - P''/|d| + 1.2e-7 t <= t, because P''/|d| >= 0.74 P / |d| >= 3.5e-7
// range_max / |d| (t <= range_max) for |d| up to 2.9: directions of ray lists are taken as given
// and need not have unit length.  In the same way every computed far value is >= t.  So
// tmin <= tmax holds as computed, with no relative slack, and the box is never culled; boxes
// grow by about 2^-21 range_max (0.05 mm at 100 m).  SlabRay holds the per-ray constants of
// that test.
struct SlabRay {
  float idx, idy, idz;   // reciprocal direction (components clamped away from zero)
  float lx, ly, lz;      // -(o + P) / d: offsets of the lo planes
  float hx, hy, hz;      // -(o - P) / d: offsets of the hi planes
};

RMH_SLAB_HD SlabRay make_slab_ray(float ox, float oy, float oz, float dx, float dy, float dz, float range_max) {
  constexpr float kMinDir = 0x1p-64f;
  SlabRay r;
  r.idx = RMH_SLAB_RECIPROCAL(fabsf(dx) > kMinDir ? dx : copysignf(kMinDir, dx));
  r.idy = RMH_SLAB_RECIPROCAL(fabsf(dy) > kMinDir ? dy : copysignf(kMinDir, dy));
  r.idz = RMH_SLAB_RECIPROCAL(fabsf(dz) > kMinDir ? dz : copysignf(kMinDir, dz));
  const float omax = fmaxf(fmaxf(fabsf(ox), fabsf(oy)), fabsf(oz));
  const float P = (omax + range_max) * 0x1p-21f + 1e-30f;
  r.lx = -((ox + P) * r.idx); r.hx = -((ox - P) * r.idx);
  r.ly = -((oy + P) * r.idy); r.hy = -((oy - P) * r.idy);
  r.lz = -((oz + P) * r.idz); r.hz = -((oz - P) * r.idz);
  return r;
}

}  // namespace rmh
