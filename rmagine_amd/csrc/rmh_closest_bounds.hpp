// Triangle distances of the closest-point walk (rmh_closest.hip): the FP64 evaluation and the
// FP32 bounds, compiled for the device and, with host stand-ins for the two approximate
// instructions, by tests/cpp/tri_bound_check.cpp and tests/cpp/closest_eval_check.cpp.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define RMH_CB_HD __host__ __device__ inline
#else
#define RMH_CB_HD inline
#endif

#if defined(__HIP_DEVICE_COMPILE__)
#define RMH_CB_RCP(x) __builtin_amdgcn_rcpf(x)
#define RMH_CB_SQRT(x) __builtin_amdgcn_sqrtf(x)
#elif !defined(RMH_CB_RCP)  // both instructions are within one ulp; the check puts such errors in
#define RMH_CB_RCP(x) (1.0f / (x))
#define RMH_CB_SQRT(x) sqrtf(x)
#endif

namespace rmh {

struct D3 { double x, y, z; };

RMH_CB_HD D3 d3(double x, double y, double z) { D3 r; r.x = x; r.y = y; r.z = z; return r; }
RMH_CB_HD D3 sub(const D3& a, const D3& b) { return d3(a.x - b.x, a.y - b.y, a.z - b.z); }
RMH_CB_HD double ddot(const D3& a, const D3& b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
RMH_CB_HD D3 madd(const D3& a, const D3& b, double s) { return d3(a.x + b.x * s, a.y + b.y * s, a.z + b.z * s); }

// Closest point of triangle (a, b, c) to p.
RMH_CB_HD D3 closest_on_triangle(const D3& p, const D3& a, const D3& b, const D3& c) {
  const D3 ab = sub(b, a), ac = sub(c, a), ap = sub(p, a);
  const double d1 = ddot(ab, ap), d2 = ddot(ac, ap);
  if (d1 <= 0.0 && d2 <= 0.0) return a;
  const D3 bp = sub(p, b);
  const double d3v = ddot(ab, bp), d4 = ddot(ac, bp);
  if (d3v >= 0.0 && d4 <= d3v) return b;
  const double vc = d1 * d4 - d3v * d2;
  if (vc <= 0.0 && d1 >= 0.0 && d3v <= 0.0) return madd(a, ab, d1 / (d1 - d3v));
  const D3 cp = sub(p, c);
  const double d5 = ddot(ab, cp), d6 = ddot(ac, cp);
  if (d6 >= 0.0 && d5 <= d6) return c;
  const double vb = d5 * d2 - d1 * d6;
  if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) return madd(a, ac, d2 / (d2 - d6));
  const double va = d3v * d6 - d5 * d4;
  if (va <= 0.0 && (d4 - d3v) >= 0.0 && (d5 - d6) >= 0.0)
    return madd(b, sub(c, b), (d4 - d3v) / ((d4 - d3v) + (d5 - d6)));
  const double den = 1.0 / (va + vb + vc);
  return madd(madd(a, ab, vb * den), ac, vc * den);
}

struct F3 {
  float x, y, z;
};

RMH_CB_HD float fdot(const F3& a, const F3& b) { return fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x)); }
RMH_CB_HD F3 fsub(const F3& a, const F3& b) { return F3{a.x - b.x, a.y - b.y, a.z - b.z}; }

// Squared distance from the query to the box [lo, hi] in FP32, within 2^-21 of the exact one:
// each difference of two floats is rounded once (2^-24 of itself, twice that when squared),
// the product and the two fmas once each.  Overflow is infinite.
RMH_CB_HD float box_d2(const F3& q, float lox, float hix, float loy, float hiy, float loz, float hiz) {
  const float dx = fmaxf(fmaxf(lox - q.x, q.x - hix), 0.0f);
  const float dy = fmaxf(fmaxf(loy - q.y, q.y - hiy), 0.0f);
  const float dz = fmaxf(fmaxf(loz - q.z, q.z - hiz), 0.0f);
  return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// What box_d2 is compared with: a box whose value exceeds it is farther than `upper` (a bound
// of the squared distance looked for; infinite: every box is walked).  Raising the bound once
// per improvement takes the place of lowering every box's value.
RMH_CB_HD float walk_bound(float upper) { return fmaf(upper, 1.0f + 0x1p-19f, 1e-36f); }

// Bounds of the squared distance from the query to the triangle with vertices A, B, C (FP32,
// relative to the query: one rounding per component).  Both are rigorous, and a few 2^-20
// apart for triangles of ordinary shape:
// * P = A + v (B - A) + w (C - A) with weights clamped to the triangle lies on it up to
//   rounding, so the distance is at most |P| + err.  With M the largest vertex component, a
//   component of P is off by at most 27 x 2^-24 M (vertex rounding 1, edges 4, the two fmas 6,
//   weights summing to at most 1 + 2^-22 16), |P| by sqrt(3) times that: err = 2^-18 M.
// * The triangle lies beyond the plane through its lowest vertex along P, so its distance is
//   at least min(P.A, P.B, P.C) / |P|: the distance itself where P is the nearest point.  The
//   products are off by three roundings each and by the vertices' rounding, together
//   4.01 x 2^-24 |P|_1 M (|P|_1 the sum of P's components); 2^-21 of that is taken off.
// Nothing is assumed of the choice of P: a poor one (overflow, NaN) only makes the lower bound
// 0 and the upper one infinite or loose.  Degenerate triangles and slivers (sine of the angle at
// A below 0.003) get the bounds 0 and infinity, so that their FP64 evaluation alone decides: it
// has no result for equal A and B and queries on C's side (0 / 0), and in slivers its rounding
// may exceed the margins, so an upper bound of theirs could drop the triangle that the
// evaluation picks.  Values near the ends of the FP32 range get the lower bound 0.
struct D2Bounds {
  float lo, hi;
};

RMH_CB_HD D2Bounds triangle_bounds(const F3& A, const F3& B, const F3& C) {
  const F3 ab = fsub(B, A), ac = fsub(C, A);
  const float d1 = -fdot(ab, A), d2 = -fdot(ac, A);
  const float e = fdot(ab, ab), f = fdot(ab, ac), g = fdot(ac, ac);
  const float d3 = d1 - e, d4 = d2 - f, d5 = d1 - f, d6 = d2 - g;
  const float vc = fmaf(d1, d4, -(d3 * d2)), vb = fmaf(d5, d2, -(d1 * d6)), va = fmaf(d3, d6, -(d5 * d4));
  // weights of B and C: inside the face, then the edges and corners that take over
  const float den = RMH_CB_RCP(va + vb + vc);
  float v = vb * den, w = vc * den;
  const float t1 = d4 - d3, t2 = d5 - d6, t = t1 * RMH_CB_RCP(t1 + t2);
  const bool on_bc = va <= 0.0f && t1 >= 0.0f && t2 >= 0.0f;
  v = on_bc ? 1.0f - t : v;
  w = on_bc ? t : w;
  const bool on_ac = vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f;
  v = on_ac ? 0.0f : v;
  w = on_ac ? d2 * RMH_CB_RCP(g) : w;
  const bool at_c = d6 >= 0.0f && d5 <= d6;
  v = at_c ? 0.0f : v;
  w = at_c ? 1.0f : w;
  const bool on_ab = vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f;
  v = on_ab ? d1 * RMH_CB_RCP(e) : v;
  w = on_ab ? 0.0f : w;
  const bool at_b = d3 >= 0.0f && d4 <= d3;
  v = at_b ? 1.0f : v;
  w = at_b ? 0.0f : w;
  const bool at_a = d1 <= 0.0f && d2 <= 0.0f;
  v = at_a ? 0.0f : v;
  w = at_a ? 0.0f : w;
  v = fminf(fmaxf(v, 0.0f), 1.0f);
  w = fminf(fmaxf(w, 0.0f), 1.0f - v);
  const F3 P{fmaf(ac.x, w, fmaf(ab.x, v, A.x)), fmaf(ac.y, w, fmaf(ab.y, v, A.y)), fmaf(ac.z, w, fmaf(ab.z, v, A.z))};
  const float low = fminf(fminf(fdot(P, A), fdot(P, B)), fdot(P, C));
  const float M = fmaxf(fmaxf(fmaxf(fabsf(A.x), fabsf(A.y)), fmaxf(fabsf(A.z), fabsf(B.x))),
                        fmaxf(fmaxf(fmaxf(fabsf(B.y), fabsf(B.z)), fmaxf(fabsf(C.x), fabsf(C.y))), fabsf(C.z)));
#ifdef RMH_CB_NO_MARGIN  // tests/cpp/tri_bound_check.cpp: the check has to find what the margins are for
  const float lo_margin = 0.0f, hi_margin = 0.0f, slack = 0.0f;
#else
  const float lo_margin = 0x1p-21f, hi_margin = 0x1p-18f, slack = 0x1p-20f;
#endif
  const float pp = fdot(P, P);
  const float m = fmaf(-lo_margin * (fabsf(P.x) + fabsf(P.y) + fabsf(P.z)), M, low), mm = m * m;
  const float u = fmaf(M, hi_margin, RMH_CB_SQRT(pp) * (1.0f + 0.5f * slack));
  const bool shaped = fmaf(e, g, -(f * f)) > 1e-5f * (e * g);
  const bool plain = shaped && m > 0.0f && pp > 1e-30f && mm > 1e-30f && mm < 1e38f;
  D2Bounds r;
  r.lo = plain ? mm * RMH_CB_RCP(pp) * (1.0f - slack) : 0.0f;
  r.hi = shaped ? fmaf(u * u, 1.0f + slack, 1e-36f) : INFINITY;
  return r;
}

}  // namespace rmh
