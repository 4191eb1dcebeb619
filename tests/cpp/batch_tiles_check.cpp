// Host check of the batched launch's tile lookup (rmagine_amd/csrc/rmh_batch_tiles.hpp, which the
// kernel compiles): launches are made for one table and run against another one of the same
// entries, as a recorded launch is after the batch was cut into other tiles.  Every tile must lie
// in the launch's entries, every tile of them that the launch has workgroups for must come up
// once, and none other.
//
// usage: batch_tiles_check  -- prints the numbers of launches and of violations.  Built with
// -DBATCH_TILES_FIXED_BASE the launch keeps the first tile of the table it was made for: that
// must violate, which shows the check can fail.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../rmagine_amd/csrc/rmh_batch_tiles.hpp"

static uint64_t state = 0x9E3779B97F4A7C15ull;
static uint32_t below(uint32_t n) {
  uint64_t z = (state += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return static_cast<uint32_t>((z ^ (z >> 31)) % n);
}

static bool tile_of(const std::vector<uint64_t>& made, const std::vector<uint64_t>& prefix, uint32_t lo, uint32_t hi,
                    uint64_t at, uint64_t& tile) {
#ifdef BATCH_TILES_FIXED_BASE
  tile = made[lo] + at;
  return tile < prefix[hi];
#else
  (void)made;
  return rmh::launch_tile(prefix.data(), lo, hi, at, tile);
#endif
}

int main() {
  long launches = 0, bad = 0;
  for (int it = 0; it < 200000; it++) {
    const uint32_t n = 1 + below(8);
    std::vector<uint64_t> made(n + 1, 0), now(n + 1, 0);
    for (uint32_t i = 0; i < n; i++) {
      const uint32_t was = below(4) == 0 ? 0 : 1 + below(20);
      made[i + 1] = made[i] + was;
      now[i + 1] = now[i] + (was == 0 || below(2) ? was : 1 + below(20));
    }
    const uint32_t split = below(n + 1);  // the groups of a two-launch batch, or one of all
    for (int g = 0; g < 3; g++) {
      const uint32_t lo = g == 1 ? split : 0, hi = g == 0 ? split : n;
      const uint64_t blocks = made[hi] - made[lo];
      std::vector<int> seen(now[n] + 1, 0);
      launches++;
      bool ok = true;
      for (uint64_t at = 0; at < blocks; at++) {
        uint64_t t = 0;
        if (!tile_of(made, now, lo, hi, at, t)) continue;
        if (t < now[lo] || t >= now[hi]) ok = false;
        else seen[t]++;
      }
      for (uint64_t t = now[lo]; t < now[hi] && ok; t++) ok = seen[t] == (t - now[lo] < blocks ? 1 : 0);
      if (!ok) bad++;
    }
  }
  std::printf("%ld %ld\n", launches, bad);
  return bad == 0 ? 0 : 1;
}
