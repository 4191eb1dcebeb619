// Host check of the ray kernels' slab test (rmagine_amd/csrc/rmh_slab.hpp, the set-up the kernels
// compile; rmh_trace.hpp: slab2) for directions that are not of unit length, as ray lists may
// hold them: lengths from 2.0 to 3.6.  As in slab_check.c, boxes are built around a point
// o + t* d of the exact ray with t* in [0, tbf] (often degenerate), and the test must neither
// cull them nor report an entry beyond t*.
//
// usage: slab_length_check [n]  -- prints the numbers of checked and culled boxes.  Built with
// -DSLAB_RECIPROCAL_WITHIN_AN_ULP the reciprocals are off by up to one ulp, as the reciprocal
// instruction's are: that must cull some.
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

#ifdef SLAB_RECIPROCAL_WITHIN_AN_ULP
static float near_reciprocal(float x) {
  const float y = 1.0f / x;
  const uint64_t k = next_u64() % 3;
  return k == 0 ? y : std::nextafterf(y, k == 1 ? INFINITY : -INFINITY);
}
#define RMH_SLAB_RECIPROCAL(x) near_reciprocal(x)
#endif
#include "../../rmagine_amd/csrc/rmh_slab.hpp"

static float coord(double scale) {
  const uint64_t k = next_u64() % 8;
  if (k == 0) return 0.0f;
  if (k == 1) return static_cast<float>(static_cast<int>(next_u64() % 41) - 20);
  return static_cast<float>((uni() * 2.0 - 1.0) * scale);
}

static double dir_comp() {
  const uint64_t k = next_u64() % 10;
  if (k == 0) return 0.0;
  if (k == 1) return (next_u64() & 1 ? 1.0 : -1.0) * 1e-30;
  if (k == 2) return (next_u64() & 1 ? 1.0 : -1.0) * 1e-7;
  return uni() * 2.0 - 1.0;
}

static float down_f(double v) { const float f = static_cast<float>(v); return f > v ? std::nextafterf(f, -INFINITY) : f; }
static float up_f(double v) { const float f = static_cast<float>(v); return f < v ? std::nextafterf(f, INFINITY) : f; }

int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 8000000;
  long culled = 0;
  for (long it = 0; it < n; it++) {
    const double oscale[4] = {1.0, 100.0, 1000.0, 10000.0};
    const float ranges[4] = {1.0f, 100.0f, 130.0f, 10000.0f};
    const double os = oscale[next_u64() % 4];
    const float o[3] = {coord(os), coord(os), coord(os)};
    double e[3], len;
    do {
      for (double& c : e) c = dir_comp();
      len = std::sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
    } while (len < 1e-3);
    const double want = 2.0 + 1.6 * uni();
    float d[3];
    for (int k = 0; k < 3; k++) d[k] = static_cast<float>(e[k] / len * want);
    const float range_max = ranges[next_u64() % 4];
    const uint64_t tk = next_u64() % 8;
    const double ts = tk == 0 ? 0.0 : (tk == 1 ? static_cast<double>(range_max) : uni() * range_max);
    const float tbf = next_u64() & 1 ? up_f(ts) : range_max;
    float lo[3], hi[3];
    for (int k = 0; k < 3; k++) {
      const double p = o[k] + ts * d[k], err = std::fabs(p) * 0x1p-50 + 0x1p-1000;
      const double ext[4] = {0.0, 1e-4, 1.0, 10.0};
      lo[k] = down_f(p - err - uni() * ext[next_u64() % 4]);
      hi[k] = up_f(p + err + uni() * ext[next_u64() % 4]);
    }
    const rmh::SlabRay r = rmh::make_slab_ray(o[0], o[1], o[2], d[0], d[1], d[2], range_max);
    const float id[3] = {r.idx, r.idy, r.idz}, lx[3] = {r.lx, r.ly, r.lz}, hx[3] = {r.hx, r.hy, r.hz};
    float tmin = 0.0f, tmax = tbf;
    for (int k = 0; k < 3; k++) {
      const float v0 = std::fmaf(lo[k], id[k], lx[k]), v1 = std::fmaf(hi[k], id[k], hx[k]);
      tmin = std::fmax(tmin, std::fmin(v0, v1));
      tmax = std::fmin(tmax, std::fmax(v0, v1));
    }
    if (!(tmin <= tmax) || !(tmin <= ts)) culled++;
  }
  std::printf("%ld %ld\n", n, culled);
  return culled == 0 ? 0 : 1;
}
