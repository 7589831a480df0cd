// Shared by the gated delta rule's token-by-token and chunked kernels.
#pragma once

#include "qh_common.h"

namespace {

// x[l] + x[l ^ 16] and x[l] + x[l ^ 32] in registers (v_permlane16/32_swap with x in both operands
// hand each lane the pair in a fixed order; the sum is the same on both lanes of a pair), instead of
// LDS permutes, whose latency sits on every token's dependent chain.
__device__ __forceinline__ float pair16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pair32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace
