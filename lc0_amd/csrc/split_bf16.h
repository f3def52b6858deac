// A float as the exact sum of three bfloat16, and products of such sums on the bfloat16 matrix instructions: the method of Henry, Tang and
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations" (ARITH 2019).
#pragma once

#include "kernel_common.h"

namespace lc0mi {

namespace {

constexpr int kParts = 3;   // of 8 significant bits each

constexpr float kMaxBf16 = 0x1.fep+127f;

// v = part[0] + part[1] + part[2] exactly (each rounded to nearest, the first one to a finite value, the remainders exact); what is below
// the least bfloat16 (2^-133) is lost. An infinity is its first part; what is not a number is so in every part. (Values beyond the
// largest bfloat16 on a path of their own: 32 positions of a 6x64 tower 139.4 -> 140.9 us for it, with selections for every value 136.2 -> 142.8.)
__device__ __forceinline__ void Split3(const floatx4& v, bf16x4 (&part)[kParts]) {
  part[0] = __builtin_convertvector(v, bf16x4);
  floatx4 rest = v - __builtin_convertvector(part[0], floatx4);
  if (__any(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))) > kMaxBf16)) {
    floatx4 first;
#pragma unroll
    for (int e = 0; e < 4; e++) first[e] = fabsf(v[e]) < INFINITY ? __builtin_amdgcn_fmed3f(v[e], -kMaxBf16, kMaxBf16) : v[e];
    part[0] = __builtin_convertvector(first, bf16x4);
    rest = v - __builtin_convertvector(part[0], floatx4);
#pragma unroll
    for (int e = 0; e < 4; e++) rest[e] = fabsf(v[e]) < INFINITY ? rest[e] : 0.0f;
  }
  part[1] = __builtin_convertvector(rest, bf16x4);
  part[2] = __builtin_convertvector(rest - __builtin_convertvector(part[1], floatx4), bf16x4);
}

// Four values from their parts, which lie `stride` elements apart. (The sum of the lower two is exact; that of the upper two can be
// beyond the largest float.)
__device__ __forceinline__ floatx4 Join3(const bf16_t* at, int stride) {
  auto part = [&](int p) { return __builtin_convertvector(*reinterpret_cast<const bf16x4*>(at + p * stride), floatx4); };
  return part(0) + (part(1) + part(2));
}

// Of the nine products of two such sums the six that reach 2^-24 of the result: part kFirst[i] of one operand by part kSecond[i] of
// the other, the smallest first and the one of the two first parts last. The latter has an accumulator of its own, so that the
// small ones are rounded at their own size.
constexpr int kProducts = 6;
constexpr int kFirst[kProducts] = {1, 2, 0, 1, 0, 0}, kSecond[kProducts] = {1, 0, 2, 0, 1, 0};

// The sum of a product whose last of the six is summed in hi and whose others in lo. Where an operand is infinite hi alone is what floats
// would give: the lower parts of the other operand are zero or of either sign, and lo is then infinite or not a number. Any finite
// value in its place does (the median of three of what is not a number is the least of the other two).
__device__ __forceinline__ float SumOfProducts(float hi, float lo) { return hi + __builtin_amdgcn_fmed3f(lo, -kMaxBf16, kMaxBf16); }

}  // namespace

}  // namespace lc0mi
