// Sums and maxima over the 64 lanes of a wavefront on the vector ALU: DPP row
// rotations within 16 lanes, v_permlane16_swap / v_permlane32_swap across
// rows. No LDS round trip as in a shuffle, and the swaps add two values at a
// time, so that eight sums cost about as much as two.
#pragma once

#include <hip/hip_runtime.h>

namespace mxg {

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <int CTRL>
__device__ inline double dpp_get(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false));
}
constexpr int ROW_ROR8 = 0x128, ROW_ROR4 = 0x124, ROW_ROR2 = 0x122, ROW_ROR1 = 0x121;

// (a, b) -> lanes 0-31 of both, lanes 32-63 of both
__device__ inline void swap32(double& a, double& b) {
  const u32x2 lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
  const u32x2 hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
  a = __hiloint2double((int)hi[0], (int)lo[0]);
  b = __hiloint2double((int)hi[1], (int)lo[1]);
}
// rows (16 lanes) a0 a1 a2 a3 and b0 b1 b2 b3 -> a0 b0 a2 b2 and a1 b1 a3 b3
__device__ inline void swap16(double& a, double& b) {
  const u32x2 lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
  const u32x2 hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
  a = __hiloint2double((int)hi[0], (int)lo[0]);
  b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double add32(double a, double b) {
  swap32(a, b);
  return a + b;
}
__device__ inline double add16(double a, double b) {
  swap16(a, b);
  return a + b;
}
// sum over each row of 16 lanes, in all of them
__device__ inline double row_sum(double v) {
  v += dpp_get<ROW_ROR8>(v);
  v += dpp_get<ROW_ROR4>(v);
  v += dpp_get<ROW_ROR2>(v);
  v += dpp_get<ROW_ROR1>(v);
  return v;
}
__device__ inline double lane_get(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// sum over the wave, in every lane
__device__ inline double wave_total(double v) {
  v = row_sum(v);
  v = add16(v, v);
  return add32(v, v);
}
// maximum over the wave, in every lane (no NaN among the values)
__device__ inline double wave_max(double v) {
  v = fmax(v, dpp_get<ROW_ROR8>(v));
  v = fmax(v, dpp_get<ROW_ROR4>(v));
  v = fmax(v, dpp_get<ROW_ROR2>(v));
  v = fmax(v, dpp_get<ROW_ROR1>(v));
  double w = v;
  swap16(v, w);
  v = fmax(v, w);
  w = v;
  swap32(v, w);
  return fmax(v, w);
}
// Sums of G values (4 or 8) over the wave: the lanes of row q = lane / 16 hold
// the sums of values q, or of values 2 q and 2 q + 1 (out[0], out[1]).
template <int G>
__device__ inline void wave_sums(const double (&v)[G], double (&out)[G / 4]) {
  static_assert(G == 4 || G == 8, "four or eight sums");
  if constexpr (G == 4) {
    out[0] = row_sum(add16(add32(v[0], v[2]), add32(v[1], v[3])));
  } else {
    const double s0 = add32(v[0], v[4]), s1 = add32(v[1], v[5]), s2 = add32(v[2], v[6]), s3 = add32(v[3], v[7]);
    out[0] = row_sum(add16(s0, s2));
    out[1] = row_sum(add16(s1, s3));
  }
}
// sum g of wave_sums' result, as a wave-uniform value
template <int G>
__device__ inline double sum_of(const double (&out)[G / 4], int g) {
  if constexpr (G == 4) return lane_get(out[0], 16 * g);
  return lane_get(out[g & 1], 16 * (g >> 1));
}

}  // namespace mxg
