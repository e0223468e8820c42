// attn_common.hpp — what the attention kernels share.
#pragma once

#include "device_common.hpp"

namespace glypr {

constexpr float ATTN_TAU = 8.0f;  // lazy-rescale threshold (natural log): p <= e^8 ~ 2981
constexpr float ATTN_LOG2E = 1.44269504f;

// Lane pairs (l, l ^ 16) and (l, l ^ 32) through gfx950's permlane swaps:
// v_permlane16_swap / v_permlane32_swap of a value with itself return, in
// every lane, the lane's own value and its partner's (in either order), all
// in VALU — no LDS round trip as with ds_bpermute.  max and + over the pair
// are order-independent, so each equals op(v, v[l ^ 16]) (resp. l ^ 32).
__device__ __forceinline__ float pair_max16(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float pair_max32(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float pair_sum16(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float pair_sum32(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

}  // namespace glypr
