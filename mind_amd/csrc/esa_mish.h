// Mish and its slope in fp32 (the algebra is described in esa_block.hip).
#pragma once
#include "esa_common.h"

namespace {

constexpr float kMishLinear = 20.f;   // above: tanh(softplus(x)) == 1 in fp32

DEVI float mish_f(float x) {
  if (x > kMishLinear) return x;
  const float w = fast_exp2(x * kLog2e);
  const float n = w * (w + 2.f);
  return x * n * __builtin_amdgcn_rcpf(n + 2.f);
}

// At x = +inf the slope is NaN, as torch's mish backward gives (inf * 0);
// x is multiplied last so that a huge negative x meets w = 0 (slope 0).
DEVI float mish_grad_f(float x) {
  if (x > kMishLinear) return x < INFINITY ? 1.f : NAN;
  const float w = fast_exp2(x * kLog2e);
  const float n = w * (w + 2.f);
  const float r = __builtin_amdgcn_rcpf(n + 2.f);
  return n * r + x * (4.f * w * (1.f + w) * (r * r));
}

}  // namespace
