// A float as the exact sum of three bfloat16, and products of such sums on the bfloat16 matrix instructions.
#pragma once

#include "kernel_common.h"

namespace lc0mi {

namespace {

constexpr int kParts = 3;   // of 8 significant bits each

// v = part[0] + part[1] + part[2] exactly (each rounded to nearest, the remainders exact), for |v| up to the largest bfloat16; what
// is below the least float is lost. An infinity is its first part.
__device__ __forceinline__ void Split3(const floatx4& v, bf16x4 (&part)[kParts]) {
  floatx4 rest = v;
#pragma unroll
  for (int p = 0; p < kParts; p++) {
    part[p] = __builtin_convertvector(rest, bf16x4);
    rest -= __builtin_convertvector(part[p], floatx4);
    if (p == 0) {
#pragma unroll
      for (int e = 0; e < 4; e++) rest[e] = rest[e] == rest[e] ? rest[e] : 0.0f;
    }
  }
}

// Four values from their parts, which lie `stride` elements apart.
__device__ __forceinline__ floatx4 Join3(const bf16_t* at, int stride) {
  floatx4 v = __builtin_convertvector(*reinterpret_cast<const bf16x4*>(at), floatx4);
#pragma unroll
  for (int p = 1; p < kParts; p++) v += __builtin_convertvector(*reinterpret_cast<const bf16x4*>(at + p * stride), floatx4);
  return v;
}

// Of the nine products of two such sums the six that reach 2^-24 of the result: part kFirst[i] of one operand by part kSecond[i] of
// the other, the smallest first and the one of the two first parts last. The latter has an accumulator of its own, so that the
// small ones are rounded at their own size.
constexpr int kProducts = 6;
constexpr int kFirst[kProducts] = {1, 2, 0, 1, 0, 0}, kSecond[kProducts] = {1, 0, 2, 0, 1, 0};

}  // namespace

}  // namespace lc0mi
