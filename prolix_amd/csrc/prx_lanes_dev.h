// Exchanges between the lanes of a wave that cost no LDS: DPP operands (4.2
// cycles) and permlane swaps (8.2), where ds_bpermute takes 6 cycles of the whole
// CU's LDS.
#pragma once

#include "prx_common.h"

namespace prx {

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
constexpr int kDppHalfMirror = 0x141;  // lane p of 8 reads lane 7 - p
constexpr int kDppXor2 = 0x4E;         // quad_perm [2, 3, 0, 1]
constexpr int kDppXor1 = 0xB1;         // quad_perm [1, 0, 3, 2]
constexpr int kDppRor8 = 0x128;        // lane l of 16 reads lane l + 8 mod 16

// x and y with their halves (of 64 lanes) or rows of 16 exchanged:
// swap32: (x.lo, y.lo), (x.hi, y.hi); swap16: the same within each half.
__device__ __forceinline__ float add_swap32(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_swap16(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same for doubles; HALF: swap32, else swap16.
template <bool HALF>
__device__ __forceinline__ double add_swap(double x, double y) {
  const auto swap = [](unsigned p, unsigned q) {
    if constexpr (HALF)
      return __builtin_amdgcn_permlane32_swap(p, q, false, false);
    else
      return __builtin_amdgcn_permlane16_swap(p, q, false, false);
  };
  const auto lo = swap((unsigned)__double2loint(x), (unsigned)__double2loint(y));
  const auto hi = swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y));
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
}  // namespace prx
