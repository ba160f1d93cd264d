// Device-side pieces shared by the dense kernels of a transformer block (block_kernels.hip, block_tail_kernel.hip).
#pragma once
#include "geometry.h"
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

// Rows of W 16-bit elements in LDS, 16-byte chunks swizzled as Tile<> has them for rows of 256 bytes and more.
template <int W>
struct RowLayout {
  static constexpr int kWidth = W;
  static_assert(W % 128 == 0, "rows start at bank 0");
  MODA_HD static int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
  MODA_HD static int off(int row, int chunk) { return row * W + ((chunk ^ swz(row)) << 3); }
};

// Packed weights: blocks of 16 features, per block the steps of 32 of the sum, per step (`item`: block * steps + step) the 16
// bytes of each lane of a wave.  First element of a lane's piece there, and of the same piece in the weight [n][32 * steps].
MODA_HD int64_t packed_piece(int64_t item, int lane) { return (item * 64 + lane) * 8; }
MODA_HD int64_t weight_piece(int block, int step, int steps, int lane) {
  return ((int64_t)(block * 16 + (lane & 15)) * steps + step) * 32 + (lane >> 4) * 8;
}

}  // namespace moda
