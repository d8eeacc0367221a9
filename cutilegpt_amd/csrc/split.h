// fp32 values as three bf16 parts, for fp32 products on the bf16 matrix cores
// (gemm_split.hip, attention_split.hip).
#pragma once

#include "common.h"

namespace cgpt {

// Operands are scaled by 2^23 on the way into their parts (exact: a power of
// two).  Every fp32 value is a multiple of 2^-149, so every part of a scaled one
// is a multiple of 2^-126 and therefore zero or a normal bf16 number: the split
// is exact for subnormal values too, whatever stands beside them.  Values of
// 2^105 and more leave bf16's range instead; an infinite or NaN part makes every
// sum that it enters infinite or NaN, which the kernels look for.
constexpr float kSplitUp = 0x1p23f, kSplitDown = 0x1p-23f;

#if defined(__HIP_DEVICE_COMPILE__)
// Four fp32 values, times `scale` (a power of two), into four bf16 values of each
// plane: x = h + m + l exactly, h = bf16(x), m = bf16(x - h), l = x - h - m
// (round to nearest; 8 + 8 + 8 significant bits).
__device__ __forceinline__ void split3(const u32x4_t& v, float scale, u32x2_t& h, u32x2_t& m, u32x2_t& l) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const float a = __uint_as_float(v[2 * p]) * scale, b = __uint_as_float(v[2 * p + 1]) * scale;
    h[p] = pack_bf16x2(a, b);
    const float ra = a - __uint_as_float(h[p] << 16), rb = b - __uint_as_float(h[p] & 0xffff0000u);
    m[p] = pack_bf16x2(ra, rb);
    l[p] = pack_bf16x2(ra - __uint_as_float(m[p] << 16), rb - __uint_as_float(m[p] & 0xffff0000u));
  }
}
#endif

// The six products of two split operands that matter, largest first: hh, hm,
// mh, mm, hl, lh as (plane of a, plane of b).  The dropped ml, lm and ll are
// below 2^-26 of the product.
constexpr int kSplitA[6] = {0, 0, 1, 1, 0, 2}, kSplitB[6] = {0, 1, 0, 1, 2, 0};

}  // namespace cgpt
