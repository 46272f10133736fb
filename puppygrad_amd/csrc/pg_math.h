// Scalar functions that kernels of several files share.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace pgk {

// 0.5 x (1 + tanh(c (x + 0.044715 x^3))), c = 0.7978846 (gelu_in_place, src/models/cpu.rs:145-152), as x times
// the logistic function of twice the argument, 1 - r for x > 0 and r else, r = e / (1 + e) with
// e = exp(-2 c |x| (1 + 0.044715 x^2)) <= 1.  The quotient gets what the sum 1 + e dropped and one correction,
// so that the error against f64 is below that of the formula with tanhf everywhere (relative to the result
// in the 2-norm 3.2, 3.4, 2.7, 1.9e-8 for |x| below 0.1, 1, 3 and above; tanhf: 3.7, 4.0, 3.6, 2.6e-8), at
// 0.7 of its time; in an epilogue of one tile per CU nothing hides that time.
__device__ __forceinline__ float gelu_share(float x) {  // r
  const float a = fabsf(x);
  const float k = -2.0f * 1.44269504f * 0.7978846f;
  const float e = __builtin_amdgcn_exp2f(a * fmaf(a * a, k * 0.044715f, k)), d = 1.0f + e;
  const float q = __builtin_amdgcn_rcpf(d), dropped = e - (d - 1.0f);
  const float r = e * q;
  return fmaf(fmaf(-d, r, e) - dropped * r, q, r);
}
__device__ __forceinline__ float gelu_tanh(float x) {
  const float r = gelu_share(x);
  return x > 0.0f ? fmaf(-fminf(x, 3.0e38f), r, x) : x * r;  // (an infinity times r = 0)
}
// The same of x + x_rest, finite, and what f32 rounds away from it.
__device__ __forceinline__ float gelu_tanh(float x, float x_rest, float& rest) {
  const float r = gelu_share(x);
  const float y = x > 0.0f ? fmaf(-x, r, x) : x * r;
  rest = x > 0.0f ? fmaf(-x, r, x - y) + (1.0f - r) * x_rest : fmaf(x, r, -y) + r * x_rest;  // (the slope is next to y / x where it counts)
  return y;
}

}  // namespace pgk
