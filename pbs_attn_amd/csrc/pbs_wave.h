// Moves between the lanes of a wavefront by row operations of the vector unit (a shuffle goes through LDS).
#pragma once
#include "pbs_common.h"

// the value of lane ^ X.  Strides 1 .. 8 are moves inside a row of sixteen lanes, 16 and 32 exchange rows.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, false);
}
// {own, partner's} in either order: what a minimum, maximum or median does not mind
struct TwoOf {
  uint32_t a, b;
};
template <int X>
__device__ __forceinline__ TwoOf with_lane_xor(uint32_t v) {
  if constexpr (X == 1) return {v, dpp_move<0xB1>(v)};                        // quad_perm 1 0 3 2
  else if constexpr (X == 2) return {v, dpp_move<0x4E>(v)};                   // quad_perm 2 3 0 1
  else if constexpr (X == 4) return {v, dpp_move<0x1B>(dpp_move<0x141>(v))};  // mirrored in eight lanes, then in four
  else if constexpr (X == 8) return {v, dpp_move<0x128>(v)};                  // rotated by eight in sixteen
  else if constexpr (X == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {r[0], r[1]};
  } else {
    static_assert(X == 32, "lane distance");
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {r[0], r[1]};
  }
}
