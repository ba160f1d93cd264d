// Device-side pieces shared by the dense kernels of a transformer block (block_kernels.hip, block_tail_kernel.hip).
#pragma once
#include "tile.h"

namespace moda {

// The exact GELU, x Phi(x) = max(x, 0) - |x| / 2 erfc(|x| / sqrt 2).  erfc(z) / 2 = exp(-z^2) t R(t) with t = 1 / (1 + 0.38 z):
// R is a degree-6 fit of erfcx(z) / 2 t over [0, 12], relative error 1.1e-6 -- three hundred times below a rounding to 11
// bits, in both tails.  A fifth of the instructions of erff, which took two thirds of the launch.  The first term is
// x - min(x, 0), which is NaN for minus infinity, as -inf (1 + erf(-inf)) is.  Both clamps are medians, which take a value
// as it comes, where fminf has it made canonical first: an instruction more each.
__device__ __forceinline__ float gelu(float x) {
  const float a = __builtin_amdgcn_fmed3f(fabsf(x), 0.f, 14.f);  // beyond, the second term is below 1e-43
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(a, 0.38f * 0.70710678f, 1.f));
  float r = -0.062705666f;
  r = __builtin_fmaf(r, t, 0.16800725f);
  r = __builtin_fmaf(r, t, -0.034941334f);
  r = __builtin_fmaf(r, t, 0.12390631f);
  r = __builtin_fmaf(r, t, 0.0903013f);
  r = __builtin_fmaf(r, t, 0.108287916f);
  r = __builtin_fmaf(r, t, 0.107143715f);
  return (x - __builtin_amdgcn_fmed3f(x, kNegInf, 0.f)) - a * t * r * fast_exp2(a * a * (-0.5f * kLog2e));
}

}  // namespace moda
