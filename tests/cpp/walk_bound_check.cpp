// Host check of the closest-point walk's box test (rmagine_amd/csrc/rmh_closest_bounds.hpp, the
// header the kernel compiles): a box is walked when box_d2 <= walk_bound(upper), and must be
// whenever `upper`, an FP32 value, is at least the squared distance from the query to the box.
// Queries reach 1e4 (and 1e19, where squares overflow), boxes are placed at gaps from 0 to 1e3,
// often with one float between plane and query.
//
// usage: walk_bound_check [n]  -- prints the numbers of checked and dropped boxes.  Built with
// -DWALK_BOUND_AS_GIVEN the bound is not raised: that must drop some.
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "../../rmagine_amd/csrc/rmh_closest_bounds.hpp"

static uint64_t state = 0x2545F4914F6CDD1Dull;
static uint64_t next_u64() {
  uint64_t z = (state += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static double uni() { return static_cast<double>(next_u64() >> 11) * 0x1p-53; }

int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 4000000;
  long dropped = 0;
  for (long it = 0; it < n; it++) {
    const double scales[4] = {1.0, 100.0, 1e4, 1e19};
    const double scale = scales[next_u64() % 4];
    float q[3], lo[3], hi[3];
    double d2 = 0.0;
    for (int k = 0; k < 3; k++) {
      q[k] = static_cast<float>((uni() * 2.0 - 1.0) * scale);
      const uint64_t mode = next_u64() % 4;
      const double gaps[4] = {0.0, uni() * 1e-3, uni() * 10.0, uni() * 1e3};
      const double ext = uni() * 5.0;
      if (next_u64() & 1) {
        lo[k] = mode == 1 && (next_u64() & 1) ? std::nextafterf(q[k], INFINITY) : static_cast<float>(q[k] + gaps[mode]);
        hi[k] = static_cast<float>(lo[k] + ext);
      } else {
        hi[k] = mode == 1 && (next_u64() & 1) ? std::nextafterf(q[k], -INFINITY) : static_cast<float>(q[k] - gaps[mode]);
        lo[k] = static_cast<float>(hi[k] - ext);
      }
      if (scale == 1e19 && (next_u64() & 1)) lo[k] = hi[k] = -q[k];  // squares near or beyond FLT_MAX
      const double d = std::fmax(std::fmax(static_cast<double>(lo[k]) - q[k], static_cast<double>(q[k]) - hi[k]), 0.0);
      d2 += d * d;  // rounded to 2^-51 at most, far inside the walk bound's margin
    }
    float upper = static_cast<float>(d2);  // infinite beyond FLT_MAX
    if (static_cast<double>(upper) < d2) upper = std::nextafterf(upper, INFINITY);
#ifdef WALK_BOUND_AS_GIVEN
    const float bound = upper;
#else
    const float bound = rmh::walk_bound(upper);
#endif
    const rmh::F3 qf{q[0], q[1], q[2]};
    if (!(rmh::box_d2(qf, lo[0], hi[0], lo[1], hi[1], lo[2], hi[2]) <= bound)) {
      if (dropped < 5) std::printf("DROPPED: box at squared distance %a, bound %a\n", d2, bound);
      dropped++;
    }
  }
  std::printf("%ld %ld\n", n, dropped);
  return dropped == 0 ? 0 : 1;
}
