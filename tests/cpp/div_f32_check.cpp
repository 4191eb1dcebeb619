// Host check of the shared-reciprocal quotient of the ray set-up: with y any approximation of
// 1 / z good to 2^-51, fma(x - z q, y, q) with q = x y is the rounded quotient x / z for x, z that are
// FP32 values, 0 < |x| <= |z|.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

static float bits(uint32_t u) {
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

int main() {
  std::mt19937 g(7);
  uint64_t bad = 0, n = 0;
  for (int i = 0; i < 2000000; i++) {
    const bool unit = i & 1;  // significands alone, and any pair of exponents
    float z = bits((unit ? 0x3f800000u : (g() % 0xfeu + 1u) << 23) | (g() & 0x7fffffu) | (g() & 0x80000000u));
    float x = bits((unit ? 0x3f000000u : (g() % 0xffu) << 23) | (g() & 0x7fffffu) | (g() & 0x80000000u));
    if (std::fabs(x) > std::fabs(z)) std::swap(x, z);
    if (x == 0.0f || z == 0.0f) continue;
    const double X = x, Z = z;
    for (int k = -2; k <= 2; k++) {  // the reciprocal off by up to two units in the last place
      double y = 1.0 / Z;
      for (int j = 0; j < (k < 0 ? -k : k); j++) y = std::nextafter(y, k < 0 ? -INFINITY : INFINITY);
      const double q = X * y;
      bad += std::fma(std::fma(-Z, q, X), y, q) != X / Z;
      bad += std::fma(std::fma(-Z, y, 1.0), y, y) != 1.0 / Z;
      n++;
    }
  }
  std::printf("%llu checked, %llu wrong\n", (unsigned long long)n, (unsigned long long)bad);
  return bad != 0;
}
