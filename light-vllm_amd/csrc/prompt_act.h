// Activations behind a prompt's projections, of what the projection's result would be in memory (PAIRS: of a gate and its value).
#pragma once
#include "common.h"

namespace lvllm {

// x / (1 + e^-x) to the last bit or so: what the product with log2(e) loses goes into the power behind it, and a Newton step takes the
// reciprocal's error.  Below -88.72 e^-x has no place in 32 bits and x / (1 + expf(-x)) is -0, as here; above, a quarter of 1 + e^-x keeps the
// reciprocal among the normal numbers, which the hardware's needs.
__device__ __forceinline__ float prompt_silu(float x) {
  const float y = -__builtin_amdgcn_fmed3f(x, -88.72f, 87.f), t = y * 1.44269504f;
  const float lost = fmaf(y, 1.92596303e-08f, fmaf(y, 1.44269504f, -t));
  float e = __builtin_amdgcn_exp2f(t);
  e = fmaf(e, lost * 0.693147181f, e);
  const float d = fmaf(e, 0.25f, 0.25f);
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  return (x * 0.25f) * (x < -88.72f ? 0.f : r);
}

template <int ACT>
__device__ __forceinline__ float prompt_act(float a, [[maybe_unused]] float b, [[maybe_unused]] float limit) {
  auto rounded = [](float f) { return BF16::to_float(BF16::from_float(f)); };
  if constexpr (ACT == LVLLM_ACT_SILU_AND_MUL) return rounded(prompt_silu(rounded(a))) * rounded(b);
  else if constexpr (ACT == LVLLM_ACT_CLAMPED_UNIT) return clamped_unit_of(rounded(a), rounded(b), limit);
  else return relu_squared_of(rounded(a));
}

}  // namespace lvllm
