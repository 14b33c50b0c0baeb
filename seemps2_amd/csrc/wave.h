// Sums over the 64 lanes of a wavefront without LDS traffic: DPP rotations
// inside the 16-lane rows, v_permlane16/32_swap across them.  A swap step
// also halves the number of values it carries, so several sums cost little
// more than one.  The summation tree is fixed (deterministic results).
#pragma once

#include "common.h"

namespace seemps {
namespace wave {

// x from the lane `CTRL` away (a DPP control that reads a valid lane everywhere).
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sum over the 16 lanes of each row, in every lane of the row.
__device__ __forceinline__ double row_sum(double x) {
  x += dpp<0x128>(x);  // row_ror:8
  x += dpp<0x124>(x);
  x += dpp<0x122>(x);
  x += dpp<0x121>(x);
  return x;
}

// Lanes 0..31: x[l] + x[l + 32]; lanes 32..63: y[l - 32] + y[l].
__device__ __forceinline__ double fold32(double x, double y) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false,
                                                   false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false,
                                                   false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Rows 0 and 2: x of the row + x of the next row; rows 1 and 3: y of the
// previous row + y of the row.
__device__ __forceinline__ double fold16(double x, double y) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(x), __double2loint(y), false,
                                                   false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(x), __double2hiint(y), false,
                                                   false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// The value of lane `l` (the same l in every lane), in every lane.
__device__ __forceinline__ double bcast(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}

// The value of lane N of each 16-lane row, in every lane of the row (one
// instruction, where readlane takes two into scalar registers).
template <int N>
__device__ __forceinline__ double row_bcast(double x) {
  return __longlong_as_double(
      __builtin_amdgcn_update_dpp(0ll, __double_as_longlong(x), 0x150 + N, 0xf, 0xf, true));
}

// Sum over the wavefront, in every lane.
__device__ __forceinline__ double sum(double x) {
  x = fold32(x, x);
  x = fold16(x, x);
  return row_sum(x);
}

// Two sums at once, in every lane.
__device__ __forceinline__ double2 sum2(double2 v) {
  double s = fold32(v.x, v.y);
  s = row_sum(fold16(s, s));
  return make_double2(bcast(s, 0), bcast(s, 32));
}

// Four sums at once, in every lane.
__device__ __forceinline__ void sum4(double2& u, double2& v) {
  const double s = row_sum(fold16(fold32(u.x, u.y), fold32(v.x, v.y)));
  u = make_double2(bcast(s, 0), bcast(s, 32));
  v = make_double2(bcast(s, 16), bcast(s, 48));
}

}  // namespace wave
}  // namespace seemps
