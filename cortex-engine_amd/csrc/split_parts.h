// fp32 operands as exact sums of three bf16 parts, for products on the bf16 matrix cores (gemm_split.hip,
// attention_split.hip).  The method: Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations" (ARITH 2019).
//
// Each part is the bf16 value nearest to what the parts before it leave: p1 + p2 + p3 == v while the third
// part's bits lie above bf16's smallest value, 2^-133 (|v| >= 2^-110).
//
// Not finite values: an infinity is +-1 in its first part, 0 in the second and itself in the third, which
// meets the other operand's first part only.  So inf * w is infinite with the right sign for every finite
// w != 0 and for an infinite one (the third parts themselves never meet), and inf * 0 is NaN; a NaN goes
// whole into the third part.  Values that round to infinity in bf16 are truncated instead.
#pragma once

#include "common.h"

namespace cortex {

struct Parts {
  bf16x8 p[3];
};

// The parts of 8 values; SPECIAL: they may be infinite, NaN or round to infinity (looked for once per
// wavefront and 8 values: with selects for each value the fp32 attention of 8 x 8 x 256 queries on 1000 keys takes
// 28.7 to 30.9 us, so 27.1).
// Every lane of the wavefront takes part.
template <bool SPECIAL>
__device__ __forceinline__ Parts split8(const float* v) {
  Parts r;
  auto put = [&r](int j, float v, bf16 h, bool whole) __attribute__((always_inline)) {
    const float r1 = v - (float)h;
    const bf16 m = whole ? (bf16)0.0f : (bf16)r1;
    r.p[0][j] = h;
    r.p[1][j] = m;
    r.p[2][j] = (bf16)(r1 - (float)m);
  };
  uint32_t mx = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (SPECIAL) mx = max(mx, __builtin_bit_cast(uint32_t, v[j]) & 0x7fffffffu);
    put(j, v[j], (bf16)v[j], false);
  }
  if (SPECIAL && __any(mx >= 0x7f7f8000u)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, v[j]), mag = bits & 0x7fffffffu;
      const uint32_t h = mag >= 0x7f800000u ? ((bits >> 16) & 0x8000u) | 0x3f80u : bits >> 16;
      put(j, v[j], mag >= 0x7f7f8000u ? __builtin_bit_cast(bf16, (uint16_t)h) : (bf16)v[j], mag >= 0x7f800000u);
    }
  }
  return r;
}

}  // namespace cortex
