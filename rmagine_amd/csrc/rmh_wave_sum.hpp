// Sums of several FP64 values over the 64 lanes of a wave: every step halves the values a lane
// carries, so 16 values take 17 exchanges instead of the 96 of one butterfly per value.  The
// exchanges are lane swaps (32 and 16 lanes apart) and data-parallel moves within rows of 16,
// which stay on the vector ALU; `__shfl_xor` goes through the LDS permute and waits for it.
// Every lane of the wave must be active.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rmh {

template <int N>
struct Acc {
  double v[N];
};

// v and u of lanes 32 (or 16) apart, added crosswise: the lower of each pair gets the sum of
// its own v and its partner's, the upper the sums of u (one swap instruction per word).
__device__ __forceinline__ double swap_add32(double v, double u) {
  const uint64_t a = __double_as_longlong(v), b = __double_as_longlong(u);
  const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(a), static_cast<uint32_t>(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b >> 32), false, false);
  return __hiloint2double(static_cast<int>(hi[0]), static_cast<int>(lo[0])) +
         __hiloint2double(static_cast<int>(hi[1]), static_cast<int>(lo[1]));
}

__device__ __forceinline__ double swap_add16(double v, double u) {
  const uint64_t a = __double_as_longlong(v), b = __double_as_longlong(u);
  const auto lo = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(a), static_cast<uint32_t>(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b >> 32), false, false);
  return __hiloint2double(static_cast<int>(hi[0]), static_cast<int>(lo[0])) +
         __hiloint2double(static_cast<int>(hi[1]), static_cast<int>(lo[1]));
}

// x of the partner at distance OFF: 8 (row rotated by 8), 4 (half row mirrored: lane i ^ 7,
// which lies in the other group of four just as i ^ 4 does), 2 and 1 (within groups of four).
template <int OFF>
__device__ __forceinline__ double partner(double x) {
  constexpr int kCtrl = OFF == 8 ? 0x128 : (OFF == 4 ? 0x141 : (OFF == 2 ? 0x4E : 0xB1));
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, kCtrl, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(0, lo, kCtrl, 0xF, 0xF, false));
}

// The same for the distances within a row, by one exchange of the half a lane does not keep.
template <int OFF>
__device__ __forceinline__ double cross_add(double v, double u) {
  const bool up = (threadIdx.x & OFF) != 0;
  return (up ? u : v) + partner<OFF>(up ? v : u);
}

// Sums of N values over the wave, each left in the lanes of one group: value g in lanes
// [g 64 / P, (g + 1) 64 / P), P = 8, 16 or 32, the least that holds N.
template <int N>
__device__ __forceinline__ double wave_sum(const Acc<N>& a) {
  constexpr int P = N <= 8 ? 8 : (N <= 16 ? 16 : 32);
  double v[P / 2];
#pragma unroll
  for (int k = 0; k < P / 2; k++) v[k] = swap_add32(k < N ? a.v[k] : 0.0, k + P / 2 < N ? a.v[k + P / 2] : 0.0);
#pragma unroll
  for (int k = 0; k < P / 4; k++) v[k] = swap_add16(v[k], v[k + P / 4]);
#pragma unroll
  for (int k = 0; k < P / 8; k++) v[k] = cross_add<8>(v[k], v[k + P / 8]);
  if constexpr (P >= 16) {
#pragma unroll
    for (int k = 0; k < P / 16; k++) v[k] = cross_add<4>(v[k], v[k + P / 16]);
  }
  double x;
  if constexpr (P == 32) x = cross_add<2>(v[0], v[1]);
  else x = v[0] + partner<2>(v[0]);
  x += partner<1>(x);
  if constexpr (P == 8) x += partner<4>(x);  // groups of four are uniform by now
  return x;
}

}  // namespace rmh
