// Cross-lane sums on the vector ALU: the butterfly v += v(lane ^ off) for off =
// 32, 16, ... without LDS permutes.  A double's permute is two ds_bpermute of
// some 60 cycles each; these take a swap or two DPP moves per step.  Within a row
// of 16 lanes, once the steps above off are done the values repeat every 2 off
// lanes, so a rotation by off finds the same partner as the exclusive or: every
// sum is the butterfly's, bit for bit.
#ifndef PLANC_AMD_WAVE_H_
#define PLANC_AMD_WAVE_H_

#include "common.h"

namespace planc {

template <int N>
__device__ inline double row_ror(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 | N, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 | N, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// v + v(lane ^ 32), v + v(lane ^ 16): the swap instructions leave the two halves
// (the even and odd rows) of v spread over all lanes.
__device__ inline double add_xor32(double v) {
  const unsigned l = (unsigned)__double2loint(v), h = (unsigned)__double2hiint(v);
  const auto lo = __builtin_amdgcn_permlane32_swap(l, l, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(h, h, false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ inline double add_xor16(double v) {
  const unsigned l = (unsigned)__double2loint(v), h = (unsigned)__double2hiint(v);
  const auto lo = __builtin_amdgcn_permlane16_swap(l, l, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// v of one (wave-uniform) lane, in every lane.
__device__ inline double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the 16 lanes of a row, in every lane of it (all lanes active).
__device__ inline double row_sum(double v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  v += row_ror<1>(v);
  return v;
}

// Sum over the wavefront, in every lane (all lanes active).
__device__ inline double wave_sum(double v) { return row_sum(add_xor16(add_xor32(v))); }

}  // namespace planc

#endif  // PLANC_AMD_WAVE_H_
