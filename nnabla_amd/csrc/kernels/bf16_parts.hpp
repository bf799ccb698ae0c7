// An fp32 number as the sum of three bf16 numbers, exactly: eight bits each, hi and mid rounded half up in magnitude.
#pragma once
#include "common.hpp"

namespace nbla_hip {

// Two numbers at a time, as the packed words of an MFMA operand.
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
  uint32_t h[2], m[2], l[2];
  const float v[2] = {a, b};
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    h[c] = (__float_as_uint(v[c]) + 0x8000u) & 0xffff0000u;
    const float r = v[c] - __uint_as_float(h[c]);
    m[c] = (__float_as_uint(r) + 0x8000u) & 0xffff0000u;
    l[c] = __float_as_uint(r - __uint_as_float(m[c]));
  }
  hi = __builtin_amdgcn_perm(h[1], h[0], 0x07060302u);
  mid = __builtin_amdgcn_perm(m[1], m[0], 0x07060302u);
  lo = __builtin_amdgcn_perm(l[1], l[0], 0x07060302u);
}

} // namespace nbla_hip
