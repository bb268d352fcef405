// Sums over the 64 lanes of a wave on the cross-lane paths of the vector unit
// (DPP and the permlane swaps), with no LDS round trip.
#pragma once

#include <hip/hip_runtime.h>

namespace dmrg {

__device__ __forceinline__ double as_d(unsigned long long u) { return __longlong_as_double((long long)u); }

template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (unsigned)u, CTRL, 0xF, 0xF, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (unsigned)(u >> 32), CTRL, 0xF, 0xF, true);
  return as_d(((unsigned long long)hi << 32) | lo);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;

// a and b summed over lane pairs 32 (16) apart: the result holds a's sums in
// the lanes with that bit clear and b's in the others
__device__ __forceinline__ double fold32(double a, double b) {
  const unsigned long long ua = (unsigned long long)__double_as_longlong(a), ub = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return as_d(((unsigned long long)hi[0] << 32) | lo[0]) + as_d(((unsigned long long)hi[1] << 32) | lo[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
  const unsigned long long ua = (unsigned long long)__double_as_longlong(a), ub = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return as_d(((unsigned long long)hi[0] << 32) | lo[0]) + as_d(((unsigned long long)hi[1] << 32) | lo[1]);
}

// Wave sums of 16 values at once, each stage halving the registers: lane l
// ends with the sum of value bits (l>>2 & 1) + 2 (l>>3 & 1) + 4 (l>>4 & 1) +
// 8 (l>>5 & 1).  A fixed order (63 instructions against 300 for 16 butterflies).
__device__ __forceinline__ double wave_sums16(const double (&v)[16], int lane) {
  double s[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) s[t] = fold32(v[t], v[t + 8]);
#pragma unroll
  for (int t = 0; t < 4; ++t) s[t] = fold16(s[t], s[t + 4]);
  const bool b3 = lane & 8, b2 = lane & 4;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const double keep = b3 ? s[t + 2] : s[t], send = b3 ? s[t] : s[t + 2];
    s[t] = keep + dpp<DPP_MIRROR>(send);
  }
  const double keep = b2 ? s[1] : s[0], send = b2 ? s[0] : s[1];
  double x = keep + dpp<DPP_HALF_MIRROR>(send);
  x += dpp<DPP_XOR2>(x);
  x += dpp<DPP_XOR1>(x);
  return x;
}
__device__ __forceinline__ int sum_index(int lane) {
  return ((lane >> 2) & 1) | ((lane >> 2) & 2) | ((lane >> 2) & 4) | ((lane >> 2) & 8);
}

// Wave sums of two values: lanes < 32 end with a's, the others with b's
__device__ __forceinline__ double wave_sums2(double a, double b) {
  double x = fold32(a, b);
  x = fold16(x, x);      // both rows of a half: the same sum
  x += dpp<DPP_MIRROR>(x);
  x += dpp<DPP_HALF_MIRROR>(x);
  x += dpp<DPP_XOR2>(x);
  x += dpp<DPP_XOR1>(x);
  return x;
}

__device__ __forceinline__ double lane_value(double x, int l) {   // wave-uniform
  const unsigned long long u = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, l), hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), l);
  return as_d(((unsigned long long)hi << 32) | lo);
}

// sums of four values over the wave
__device__ __forceinline__ void wave_sums4(double& a, double& b, double& c, double& d) {
  double t = fold16(fold32(a, c), fold32(b, d));
  t += dpp<DPP_MIRROR>(t);
  t += dpp<DPP_HALF_MIRROR>(t);
  t += dpp<DPP_XOR2>(t);
  t += dpp<DPP_XOR1>(t);
  a = lane_value(t, 0);
  b = lane_value(t, 16);
  c = lane_value(t, 32);
  d = lane_value(t, 48);
}

}  // namespace dmrg
