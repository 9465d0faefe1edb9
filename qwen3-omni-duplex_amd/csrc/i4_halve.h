// Halving butterfly: many wave sums at once, each in the order in which group_sum adds.
// A step adds the same lane pairs as group_sum's step over that lane bit, but every lane
// keeps half of the values, so 64 sums cost 2.8 instructions each and end one per lane.
#pragma once

#include "i4_common.h"

namespace i4 {

// One step over lane bit BIT: the lane with the bit clear ends with a(l) + a(l ^ bit),
// the lane with it set with b(l) + b(l ^ bit) -- the sums group_sum forms at that step.
template <int BIT> __device__ inline float from_xor(float v) {
  if constexpr (BIT == 0) return dpp_mov<0xB1>(v);  // quad_perm [1,0,3,2]
  else if constexpr (BIT == 1) return dpp_mov<0x4E>(v);  // quad_perm [2,3,0,1]
  else if constexpr (BIT == 2) return dpp_mov<0x1B>(dpp_mov<0x141>(v));  // 7 - l, then 3 - l
  else if constexpr (BIT == 3) return dpp_mov<0x128>(v);  // row_ror:8
  else if constexpr (BIT == 4)
    return __builtin_bit_cast(
        float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
  else
    return __builtin_bit_cast(
        float, __builtin_amdgcn_ds_bpermute(((int)__lane_id() ^ 32) << 2,
                                            __builtin_bit_cast(int, v)));
}
template <int BIT> __device__ inline float halve(float a, float b, int lane) {
  const bool hi = (lane >> BIT) & 1;
  return (hi ? b : a) + from_xor<BIT>(hi ? a : b);
}

// rows 0..7 of one token over lane bits 0..2: lane l ends with row l & 7
__device__ inline float halve_rows(const float (&v)[8], int lane) {
  float u[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = halve<0>(v[2 * i], v[2 * i + 1], lane);
  return halve<2>(halve<1>(u[0], u[1], lane), halve<1>(u[2], u[3], lane), lane);
}

// 8 tokens' halve_rows results over lane bits 3..5: lane l ends with row l & 7 of token l >> 3
__device__ inline float halve_tokens(const float (&v)[8], int lane) {
  float u[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = halve<3>(v[2 * i], v[2 * i + 1], lane);
  return halve<5>(halve<4>(u[0], u[1], lane), halve<4>(u[2], u[3], lane), lane);
}

}  // namespace i4
