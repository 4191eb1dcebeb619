// Which tile of a batch table a workgroup of a launch casts.  Shared by the batched kernel
// (rmh_simulate.hip) and its host check (tests/cpp/batch_tiles_check.cpp).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define RMH_BT_HD __host__ __device__ inline
#else
#define RMH_BT_HD inline
#endif

namespace rmh {

// Entry i of the table holds the tiles [prefix[i], prefix[i + 1]); `at` counts the tiles of the
// entries [lo, hi) from the first one.  A launch recorded into a graph keeps lo, hi and its
// counts while rmh_batch_set_params may cut the table into other tiles, so both ends come from
// the table as it is: the tile lies in [prefix[lo], prefix[hi]), or there is none (false).
RMH_BT_HD bool launch_tile(const uint64_t* prefix, uint32_t lo, uint32_t hi, uint64_t at, uint64_t& tile) {
  tile = prefix[lo] + at;
  return tile < prefix[hi];
}

}  // namespace rmh
