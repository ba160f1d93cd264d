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

// Layer norm of 256 / LPR rows, LPR lanes a row with CH pieces of eight each (block_kernels.hip).
template <typename T, int LPR, int CH>
__device__ __forceinline__ void layer_norm_rows(unsigned block, const uint16_t* x, const uint16_t* weight, const uint16_t* bias, float eps, uint16_t* y,
                                                int rows, int dim) {
  const int tid = threadIdx.x, sub = tid % LPR;
  const int row = (int)block * (256 / LPR) + tid / LPR;
  if (row >= rows) return;  // whole lane groups leave together
  auto sum = [](float v) {
#pragma unroll
    for (int s = LPR / 2; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
    return v;
  };
  auto load8 = [](const uint16_t* p, float (&f)[8]) {
    const i32x4 v = *reinterpret_cast<const i32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; i++) unpack2<T>(v[i], f[2 * i], f[2 * i + 1]);
  };
  float f[CH][8], s = 0.f;
#pragma unroll
  for (int c = 0; c < CH; c++) {
    const int e = (c * LPR + sub) * 8;
#pragma unroll
    for (int i = 0; i < 8; i++) f[c][i] = 0.f;
    if (e < dim) load8(x + (int64_t)row * dim + e, f[c]);
#pragma unroll
    for (int i = 0; i < 8; i++) s += f[c][i];
  }
  const float mean = sum(s) / dim;
  float v = 0.f;
#pragma unroll
  for (int c = 0; c < CH; c++)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float d = f[c][i] - mean;
      if ((c * LPR + sub) * 8 < dim) v = __builtin_fmaf(d, d, v);
    }
  const float rstd = rsqrtf(sum(v) / dim + eps);
#pragma unroll
  for (int c = 0; c < CH; c++) {
    const int e = (c * LPR + sub) * 8;
    if (e >= dim) continue;
    float w[8], b[8];
    load8(weight + e, w);
    load8(bias + e, b);
    i32x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++)
      o[i] = pack2<T>((f[c][2 * i] - mean) * rstd * w[2 * i] + b[2 * i], (f[c][2 * i + 1] - mean) * rstd * w[2 * i + 1] + b[2 * i + 1]);
    *reinterpret_cast<i32x4*>(y + (int64_t)row * dim + e) = o;
  }
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
