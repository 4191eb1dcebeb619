// Host check of normal_radius (rmagine_amd/csrc/rmh_noise_draw.hpp), the radius of the
// Box-Muller draw: every draw m = 1 .. 2^24 against sqrt(-2 log u) in long double; prints the
// largest relative error of it and of the FP64 formula sqrt(-2 log u) of libm.
#include <cstdio>

#include "../../rmagine_amd/csrc/rmh_noise_draw.hpp"

int main() {
  double worst = 0.0, libm = 0.0;
  uint32_t n = 0;
  for (uint32_t m = 1; m <= (1u << 24); m++, n++) {
    const double a = rmh::normal_radius(m);
    const double u = m * 0x1p-24;
    const long double ref = sqrtl(-2.0L * logl(static_cast<long double>(u)));
    if (ref == 0.0L) {
      if (a != 0.0) return 1;
      continue;
    }
    const double e = static_cast<double>(fabsl((a - ref) / ref));
    const double e2 = static_cast<double>(fabsl((std::sqrt(-2.0 * std::log(u)) - ref) / ref));
    if (!(e <= worst)) worst = e;
    if (!(e2 <= libm)) libm = e2;
  }
  std::printf("%u %.3e %.3e\n", n, worst, libm);
  return worst < 1e-15 ? 0 : 1;
}
