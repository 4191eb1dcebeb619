// Host check of the closest-point walk's FP32 bounds (rmagine_amd/csrc/rmh_closest_bounds.hpp,
// the header the kernel compiles): for random queries, triangles and boxes the bounds must
// enclose the squared distance computed in FP64.  The reciprocal and square root instructions
// are stood in for by correctly rounded results moved by -1, 0 or 1 ulp.  Scales reach from
// 1e-3 to 1e5, distances from zero (queries on a vertex, an edge, the face) to far away, and
// shapes include slivers and degenerate triangles.
//
// usage: tri_bound_check [n]  -- prints the numbers of checked and violating cases; exit
// status 0 when there is none.  Built with -DRMH_CB_NO_MARGIN it must find violations.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

static uint64_t state = 0x9E3779B97F4A7C15ull;
static uint64_t next_u64() {
  uint64_t z = (state += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static double uni() { return static_cast<double>(next_u64() >> 11) * 0x1p-53; }

static float moved(float x) {
  if (!std::isfinite(x) || x == 0.0f) return x;
  const uint64_t k = next_u64() % 3;
  return k == 0 ? std::nextafterf(x, -INFINITY) : (k == 1 ? std::nextafterf(x, INFINITY) : x);
}
#define RMH_CB_RCP(x) moved(1.0f / (x))
#define RMH_CB_SQRT(x) moved(sqrtf(x))
#include "../../rmagine_amd/csrc/rmh_closest_bounds.hpp"

struct D3 { double x, y, z; };
static D3 sub(D3 a, D3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
static double dot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
static D3 cross(D3 a, D3 b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }

static double segment_d2(D3 p, D3 a, D3 b) {
  const D3 ab = sub(b, a), ap = sub(p, a);
  const double l = dot(ab, ab);
  double t = l > 0 ? dot(ap, ab) / l : 0;
  t = t < 0 ? 0 : (t > 1 ? 1 : t);
  const D3 d = {ap.x - t * ab.x, ap.y - t * ab.y, ap.z - t * ab.z};
  return dot(d, d);
}

static double triangle_d2(D3 p, D3 a, D3 b, D3 c) {
  double best = std::fmin(std::fmin(segment_d2(p, a, b), segment_d2(p, b, c)), segment_d2(p, c, a));
  const D3 n = cross(sub(b, a), sub(c, a));
  const double nn = dot(n, n);
  if (nn > 0 && dot(cross(sub(b, a), sub(p, a)), n) >= 0 && dot(cross(sub(c, b), sub(p, b)), n) >= 0 &&
      dot(cross(sub(a, c), sub(p, c)), n) >= 0) {
    const double h = dot(sub(p, a), n);
    best = std::fmin(best, h * h / nn);
  }
  return best;
}

int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 4000000;
  long bad = 0;
  for (long it = 0; it < n; it++) {
    const double where = std::pow(10.0, uni() * 5.0 - 1.0), size = std::pow(10.0, uni() * 5.0 - 3.0);
    float v[3][3], q[3];
    const uint64_t shape = next_u64() % 8;
    for (int k = 0; k < 3; k++) {
      const double c = (uni() * 2 - 1) * where;
      for (int i = 0; i < 3; i++) v[i][k] = static_cast<float>(c + (uni() * 2 - 1) * size);
    }
    if (shape == 0)  // sliver: C close to the line A B
      for (int k = 0; k < 3; k++) v[2][k] = static_cast<float>(v[0][k] + 0.4 * ((double)v[1][k] - v[0][k]) + (uni() - 0.5) * size * 1e-4);
    if (shape == 1)  // degenerate: two vertices, or all three, the same
      for (int k = 0; k < 3; k++) { v[2][k] = v[0][k]; if (next_u64() % 4 == 0) v[1][k] = v[0][k]; }
    // the query: a point of the triangle's plane (weights in or out of it), moved off it
    const uint64_t place = next_u64() % 6;
    double a = uni(), b = uni();
    if (place == 0) { a = 0; b = 0; }
    if (place == 1) b = 0;
    if (place == 2) { a = 3 * uni() - 1; b = 3 * uni() - 1; }
    const double away = place == 3 ? 0.0 : size * std::pow(10.0, uni() * 6.0 - 4.0);
    for (int k = 0; k < 3; k++)
      q[k] = static_cast<float>(v[0][k] + a * ((double)v[1][k] - v[0][k]) + b * ((double)v[2][k] - v[0][k]) + (uni() * 2 - 1) * away);
    const D3 p = {q[0], q[1], q[2]};
    const D3 t[3] = {{v[0][0], v[0][1], v[0][2]}, {v[1][0], v[1][1], v[1][2]}, {v[2][0], v[2][1], v[2][2]}};
    const double d2 = triangle_d2(p, t[0], t[1], t[2]);
    // rounding of the FP64 distance itself: 2^-46 of the largest vertex vector times the distance
    const double reach = std::sqrt(std::fmax(dot(sub(t[0], p), sub(t[0], p)), std::fmax(dot(sub(t[1], p), sub(t[1], p)), dot(sub(t[2], p), sub(t[2], p)))));
    const double tol = 0x1p-46 * reach * (std::sqrt(d2) + 0x1p-46 * reach);
    const rmh::F3 qf{q[0], q[1], q[2]};
    const rmh::D2Bounds r = rmh::triangle_bounds(rmh::fsub(rmh::F3{v[0][0], v[0][1], v[0][2]}, qf),
                                                 rmh::fsub(rmh::F3{v[1][0], v[1][1], v[1][2]}, qf),
                                                 rmh::fsub(rmh::F3{v[2][0], v[2][1], v[2][2]}, qf));
    if (r.lo > d2 + tol || r.hi < d2 - tol) {
      if (bad < 5) std::printf("VIOLATION: triangle, bounds %a %a, squared distance %a\n", r.lo, r.hi, d2);
      bad++;
    }
    // the triangle's box: kept whenever `upper` reaches its distance
    float lo[3], hi[3];
    double box = 0;
    for (int k = 0; k < 3; k++) {
      lo[k] = std::fminf(v[0][k], std::fminf(v[1][k], v[2][k]));
      hi[k] = std::fmaxf(v[0][k], std::fmaxf(v[1][k], v[2][k]));
      const double d = std::fmax(std::fmax((double)lo[k] - q[k], (double)q[k] - hi[k]), 0.0);
      box += d * d;
    }
    float upper = static_cast<float>(box);
    if (static_cast<double>(upper) < box) upper = std::nextafterf(upper, INFINITY);
#ifdef RMH_CB_NO_MARGIN
    const float limit = upper;
#else
    const float limit = rmh::walk_bound(upper);
#endif
    if (rmh::box_d2(qf, lo[0], hi[0], lo[1], hi[1], lo[2], hi[2]) > limit) {
      if (bad < 5) std::printf("VIOLATION: box at squared distance %a dropped\n", box);
      bad++;
    }
  }
  std::printf("%ld %ld\n", n, bad);
  return bad == 0 ? 0 : 1;
}
