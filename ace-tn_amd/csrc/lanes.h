// Device helpers shared by the small linear algebra kernels: values and sums
// across the lanes of a wave, and refined reciprocals.
#pragma once
#include <hip/hip_runtime.h>

namespace acetn {

// x of one lane, in a scalar register
__device__ __forceinline__ double lane_value(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// ---- sums over lanes by data-parallel moves (no LDS round trip); every lane
// gets the same bits
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sum16(double x) {
  x += dpp_mov<0xB1>(x);   // lane ^ 1
  x += dpp_mov<0x4E>(x);   // lane ^ 2
  x += dpp_mov<0x141>(x);  // the other quad of the 8
  x += dpp_mov<0x140>(x);  // the other half of the row of 16
  return x;
}
// sum over each half-wave of 32
__device__ __forceinline__ double sum32(double x) {
  x = sum16(x);
  const unsigned lo = __double2loint(x), hi = __double2hiint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __hiloint2double(b[0], a[0]) + __hiloint2double(b[1], a[1]);
}
__device__ __forceinline__ double sum64(double x) {
  x = sum32(x);
  const unsigned lo = __double2loint(x), hi = __double2hiint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __hiloint2double(b[0], a[0]) + __hiloint2double(b[1], a[1]);
}

// 1/sqrt(x) and 1/x from the hardware approximations with two Newton steps
// (a few ulps: the reflectors are orthogonal to that much)
__device__ __forceinline__ double rsqrt_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * x;
  y = y * fma(-h * y, y, 1.5);
  return y * fma(-h * y, y, 1.5);
}
__device__ __forceinline__ double rcp_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// NC values (a multiple of 4, at most 16) summed over the wave's lanes at once:
// each exchange of half-waves and of rows sums two values, so every lane ends
// with NC / 4 totals in k, and lane l's k[t] is that of value 4 t + lanes_of(l).
__device__ __forceinline__ double swap32_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
// lo: the even rows of 16 of a, each followed by the row of b there; hi: the
// odd ones; for a = b, the two rows of a half-wave, each in both places
__device__ __forceinline__ void swap16(double a, double b, double& lo, double& hi) {
  const auto x = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  lo = __hiloint2double(y[0], x[0]);
  hi = __hiloint2double(y[1], x[1]);
}
__device__ __forceinline__ double swap16_sum(double a, double b) {
  double lo, hi;
  swap16(a, b, lo, hi);
  return lo + hi;
}
__device__ __forceinline__ int lanes_of(int lane) {
  const int row = lane >> 4;  // rows 0..3 hold values 0, 2, 1, 3 of a group of four
  return row == 1 ? 2 : row == 2 ? 1 : row;
}
template <int NC>
__device__ __forceinline__ void sum64_many(const double (&g)[NC], double (&k)[NC / 4]) {
#pragma unroll
  for (int t = 0; t < NC / 4; ++t)
    k[t] = sum16(swap16_sum(swap32_sum(g[4 * t], g[4 * t + 1]), swap32_sum(g[4 * t + 2], g[4 * t + 3])));
}

}  // namespace acetn
