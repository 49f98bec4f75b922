// Activations behind a prompt's projections, of what the projection's result would be in memory (PAIRS: of a gate and its value).
#pragma once
#include "common.h"

namespace lvllm {

// x / (1 + e^-x) to the last bit or so: what the product with log2(e) loses goes into the power behind it, and a Newton step takes the
// reciprocal's error.  The power is taken between +-87; below, the sigmoid is 0 to any bit that x could bring back.
__device__ __forceinline__ float prompt_silu(float x) {
  const float y = -__builtin_amdgcn_fmed3f(x, -87.f, 87.f), t = y * 1.44269504f;
  const float lost = fmaf(y, 1.92596303e-08f, fmaf(y, 1.44269504f, -t));
  float e = __builtin_amdgcn_exp2f(t);
  e = fmaf(e, lost * 0.693147181f, e);
  const float d = 1.f + e;
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  return x * (x < -87.f ? 0.f : r);
}

template <int ACT>
__device__ __forceinline__ float prompt_act(float a, [[maybe_unused]] float b, [[maybe_unused]] float limit) {
  auto rounded = [](float f) { return BF16::to_float(BF16::from_float(f)); };
  if constexpr (ACT == LVLLM_ACT_SILU_AND_MUL) return rounded(prompt_silu(rounded(a))) * rounded(b);
  else if constexpr (ACT == LVLLM_ACT_CLAMPED_UNIT) return clamped_unit_of(rounded(a), rounded(b), limit);
  else return relu_squared_of(rounded(a));
}

}  // namespace lvllm
