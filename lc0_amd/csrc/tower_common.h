// What the two resident-tower kernels share (resident_tower.hip, resident_tower_f32.hip).
#pragma once

#include "kernel_common.h"

namespace lc0mi {

namespace {

constexpr int kPlanes = 128;              // the 112 input planes, padded

// The tower's activations: mish and relu.
template <typename F>
__device__ __forceinline__ void TowerAct(int act, F&& f) {
  if (act == kActMish) f([](float v) { return ActMish(v); });
  else f([](float v) { return v > 0.0f ? v : 0.0f; });
}

// Sum over the 32 lanes of each half of a wave, in the upper 16 of them.
__device__ __forceinline__ float Sum32(float v) {
  v += DppMove<0xB1>(v);
  v += DppMove<0x4E>(v);
  v += DppMove<0x141>(v);
  v += DppMove<0x140>(v);   // mirrored within 16
  v += DppMove<0x142>(v);   // the row of lanes before
  return v;
}

}  // namespace

}  // namespace lc0mi
