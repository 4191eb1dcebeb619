// Host check of what the closest-point walk takes from a triangle's FP32 upper bound
// (rmagine_amd/csrc/rmh_closest_bounds.hpp, the header the kernel compiles): the walk drops
// whatever lies beyond it, so the FP64 evaluation that names the result must not give that
// triangle a larger distance, or none (NaN).  Random triangles of all shapes (two or three equal
// vertices, vertices a few bits apart, slivers, ordinary ones) of sizes from 1e-9 to 1e3, near
// the origin or far from it, with queries on them, beside them and up to 1e6 away; the
// reciprocal and square root instructions are stood in for by correctly rounded results moved
// by -1, 0 or 1 ulp.
//
// usage: closest_eval_check [n]  -- prints the numbers of checked triangles, of finite upper
// bounds among the well-shaped ones, and of violations; exit status 0 when there is none of the last.
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

int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 6000000;
  long finite = 0, bad = 0;
  for (long it = 0; it < n; it++) {
    const double size = std::pow(10.0, uni() * 12 - 9), where = uni() < 0.3 ? 0.0 : std::pow(10.0, uni() * 8 - 3);
    float v[3][3], q[3];
    for (int k = 0; k < 3; k++) {
      const double c = (uni() * 2 - 1) * where;
      for (int i = 0; i < 3; i++) v[i][k] = static_cast<float>(c + (uni() * 2 - 1) * size);
    }
    const uint64_t shape = next_u64() % 10;
    const double thin = std::pow(10.0, -9.0 * uni());
    for (int k = 0; k < 3; k++) {
      const float near = static_cast<float>((uni() - 0.5) * size * thin);
      if (shape == 0) v[2][k] = static_cast<float>(v[0][k] + 0.4 * ((double)v[1][k] - v[0][k]) + near);
      if (shape == 1 || shape == 4) v[1][k] = v[0][k];
      if (shape == 2 || shape == 4) v[2][k] = v[0][k];
      if (shape == 3) v[2][k] = v[1][k];
      if (shape == 5) v[1][k] = v[0][k] + near;
      if (shape == 6) v[2][k] = v[0][k] + near;
      if (shape == 7) v[2][k] = v[1][k] + near;
    }
    double a = 3 * uni() - 1, b = 3 * uni() - 1;
    const uint64_t place = next_u64() % 4;
    if (place == 0) a = b = 0.0;
    if (place == 1) b = 0.0;
    const double away = place == 3 ? 0.0 : (uni() < 0.5 ? std::pow(10.0, uni() * 14 - 8) : size * std::pow(10.0, uni() * 6 - 4));
    for (int k = 0; k < 3; k++)
      q[k] = static_cast<float>(v[0][k] + a * ((double)v[1][k] - v[0][k]) + b * ((double)v[2][k] - v[0][k]) +
                                (uni() * 2 - 1) * away);
    const rmh::D3 p = rmh::d3(q[0], q[1], q[2]);
    const rmh::D3 c = rmh::closest_on_triangle(p, rmh::d3(v[0][0], v[0][1], v[0][2]), rmh::d3(v[1][0], v[1][1], v[1][2]),
                                               rmh::d3(v[2][0], v[2][1], v[2][2]));
    const double d2 = rmh::ddot(rmh::sub(c, p), rmh::sub(c, p));
    const rmh::F3 qf{q[0], q[1], q[2]};
    const rmh::D2Bounds r = rmh::triangle_bounds(rmh::fsub(rmh::F3{v[0][0], v[0][1], v[0][2]}, qf),
                                                 rmh::fsub(rmh::F3{v[1][0], v[1][1], v[1][2]}, qf),
                                                 rmh::fsub(rmh::F3{v[2][0], v[2][1], v[2][2]}, qf));
    if (shape > 7 && std::isfinite(r.hi)) finite++;
    if (std::isfinite(r.hi) && !(d2 <= r.hi)) {
      if (bad < 5)
        std::printf("VIOLATION: triangle %a %a %a  %a %a %a  %a %a %a query %a %a %a: bound %a, FP64 %a\n", v[0][0], v[0][1],
                    v[0][2], v[1][0], v[1][1], v[1][2], v[2][0], v[2][1], v[2][2], q[0], q[1], q[2], r.hi, d2);
      bad++;
    }
  }
  std::printf("%ld %ld %ld\n", n, finite, bad);
  return bad == 0 ? 0 : 1;
}
