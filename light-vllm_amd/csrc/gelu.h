#pragma once
#include "common.h"

namespace lvllm {

// x Phi(x): Phi as a sigmoid of an odd polynomial, which a least-maximum fit gave (largest error of the result 6.7e-8 before any rounding; with those of
// 32 bits 1.0e-7 for x < 0, 4.9e-7 up to 4, 5.9e-7 up to 8, where x / 2 (1 + erf) has 0.8e-7, 2.9e-7 and 4.5e-7).  13 instructions; erff is 40.
__device__ __forceinline__ float gelu_of(float x) {
  const float t = x * x;
  float p = 5.20991372e-09f;
  p = fmaf(p, t, -3.85045217e-07f);
  p = fmaf(p, t, 1.14524335e-05f);
  p = fmaf(p, t, -1.59389438e-04f);
  p = fmaf(p, t, -9.55928466e-05f);
  p = fmaf(p, t, 1.04838581e-01f);
  p = fmaf(p, t, 2.30220720f);
  return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-x * p));
}
}  // namespace lvllm
