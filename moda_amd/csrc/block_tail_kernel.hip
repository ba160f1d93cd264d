// Everything a transformer block does with a row between two attention calls, in one launch: output projection and
// residual, layer norm, MLP with exact GELU and residual, layer norm and the projections of the next block.  All of it is
// local to a row, so a workgroup takes BM rows through the whole chain; what one step hands to the next stays in
// registers and LDS.  As separate launches (block_kernels.hip) the same rows went to memory and back six times, the
// hidden activations of the MLP, four times as wide, among them: 12 608 rows of width 256 took 69 us in seven launches
// (projection 9, norm 6, MLP 23 + 15, norm 6, next projections 10.5), here 33 - 34.
//
// Eight waves share the BM rows and divide the features of every product.  The weights sit on the matrix instruction's A
// side (M = features) and go from memory (L2 after the first workgroup of an XCD) straight into the registers that it
// reads: no two waves of a workgroup read the same weight, so LDS would only add a trip.  The rows sit on the B side
// (N = rows) and come from LDS, where all waves read them.  A lane ends up with four consecutive features of a row.
//
// 64 rows where they give each compute unit a workgroup, else 32: a compute unit takes in 64 bytes of weights a cycle, and with
// 32 rows it waits for them.  (Two workgroups of 32 rows a compute unit instead: 48 us.)
//
// What bounds it, per 64 rows at width 256, hidden 1024, a next block with 384 projected features, measured cycles of 63 k: the
// MLP's products 21 k (16 k of matrix instructions; the rows' operands take all of LDS's 128 bytes a cycle there, and the
// weights all of the 64 from L2), its activation 9.4 k, waiting for each other 4 k; rows in 5 k, the two projections 9 k, norms
// and residuals 11 k, rows out 5 k.  With the activation of a chunk beside the second product of the chunk before, an
// eighth of it after each step, the two waves of a SIMD cover each other: 34.7 -> 33.5 us, 64 x 197 tokens through twelve blocks
// 571 -> 556, 16 x 197 417 -> 406.  Beside the next chunk's first product, or with the two waves of a SIMD half a chunk apart, it
// needs more registers than there are (72 spilled, 44 us; with half the weights in flight 37).
#include "block_tail.h"

namespace moda {

// Weights [n][k] into the order in which the products above read them: blocks of 16 features, per block the steps of 32 of
// the sum, per step the 1 KB of a wave's A operand, lane by lane.  In their own order a wave's load touches sixteen rows in each
// quarter of its lanes, sixteen cache lines where packed it touches two, and a compute unit takes in 13 bytes a cycle instead
// of 64 (12 608 rows, width 256: 61 us, packed 42 at the time).  Twelve blocks are packed in one launch of 7.3 us.
// The last row of workgroups fills the GELU table (see activated): bf16 values from 2^-17 to 16, then their negatives.
constexpr int kPackMatrices = 96;
struct PackArgs {
  int n;
  float* gelu_table;
  struct Matrix {
    const uint16_t* w;
    uint16_t* to;
    int blocks, steps;
  } m[kPackMatrices];
};
// Workgroup x of matrix y, or y = a.n: of the table, filled by `table_blocks` of them
__device__ __forceinline__ void pack_weights(const PackArgs& a, int x, int y, int table_blocks) {
  if (y == a.n) {
    for (int i = x * 256 + threadIdx.x; i < kGeluTable; i += table_blocks * 256) {
      const int bits = (kGeluFirst + i % kGeluHalf) | (i < kGeluHalf ? 0 : 0x8000);
      float v, g, none;
      unpack2<BF16>(bits, v, none);
      unpack2<BF16>(pack2<BF16>(gelu(v), 0.f), g, none);
      a.gelu_table[i] = g / v;
    }
    return;
  }
  const PackArgs::Matrix m = a.m[y];
  const int lane = threadIdx.x & 63, item = x * 4 + (threadIdx.x >> 6);
  if (item >= m.blocks * m.steps) return;
  const int blk = item / m.steps, ks = item - blk * m.steps;
  const i32x4 v = *reinterpret_cast<const i32x4*>(m.w + weight_piece(blk, ks, m.steps, lane));
  *reinterpret_cast<i32x4*>(m.to + packed_piece(item, lane)) = v;
}
__global__ __launch_bounds__(256) void pack_weights_kernel(const PackArgs a) { pack_weights(a, blockIdx.x, blockIdx.y, gridDim.x); }

// ... and the layer norm of a stack's input, which neither waits for the other: one launch less at the start of a pass.  Both only move
// memory.  Six blocks of width 128: 64 x 50 tokens 108.9 -> 106.1 us, 36 x 197 124.7 -> 121.3; twelve of 256 on 64 x 197 513 -> 511.
struct NormArgs {
  const uint16_t *x, *w, *b;
  uint16_t* y;
  float eps;
  int rows, dim, blocks;
};
template <typename T, int LPR>
__global__ __launch_bounds__(256) void pack_and_norm_kernel(const PackArgs a, const NormArgs n, int pack_blocks) {
  const int block = (int)blockIdx.x - n.blocks;
  if (block < 0)
    layer_norm_rows<T, LPR, 1>(blockIdx.x, n.x, n.w, n.b, n.eps, n.y, n.rows, n.dim);
  else
    pack_weights(a, block % pack_blocks, block / pack_blocks, pack_blocks);
}

namespace {

template <typename T, int C, int NB, bool POST>
hipError_t launch_tail_t(const TailArgs& a, hipStream_t stream) {
  constexpr int BM = 16 * NB, HC = 256;
  constexpr size_t smem = table_bytes<T>() + (size_t)BM * (C + (C > 2 * HC ? C : 2 * HC)) * sizeof(uint16_t);
  static LdsAttrState attr;
  const hipError_t e = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&block_tail_kernel<T, C, NB, POST>), smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((block_tail_kernel<T, C, NB, POST>), dim3((unsigned)((a.rows + BM - 1) / BM)), dim3(512), smem, stream, a);
  return hipGetLastError();
}

template <typename T, int C>
hipError_t launch_tail_c(const TailArgs& a, bool post, int cus, hipStream_t stream) {
  if (block_tail_rows(a.rows, cus) == 32) return post ? launch_tail_t<T, C, 2, true>(a, stream) : launch_tail_t<T, C, 2, false>(a, stream);
  return post ? launch_tail_t<T, C, 4, true>(a, stream) : launch_tail_t<T, C, 4, false>(a, stream);
}

template <typename T>
hipError_t launch_tail(const TailArgs& a, int width, bool post, int cus, hipStream_t stream) {
  switch (width) {
    case 128: return launch_tail_c<T, 128>(a, post, cus, stream);
    case 256: return launch_tail_c<T, 256>(a, post, cus, stream);
    case 384: return launch_tail_c<T, 384>(a, post, cus, stream);
    case 512: return launch_tail_c<T, 512>(a, post, cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_layer_norm(int dtype, int64_t rows, int64_t dim, const void* x, const void* weight, const void* bias, float eps, void* y,
                             hipStream_t stream);  // block_kernels.hip

hipError_t launch_pack_weights(const moda_hip_weight* w, int n, float* gelu_table, const moda_hip_norm_rows* norm, hipStream_t stream) {
  for (int first = 0; first < n; first += kPackMatrices) {
    PackArgs a = {};
    int64_t most = 0;
    const int count = n - first < kPackMatrices ? n - first : kPackMatrices;
    for (int i = 0; i < count; i++) {
      const moda_hip_weight& x = w[first + i];
      a.m[i] = PackArgs::Matrix{(const uint16_t*)x.w, (uint16_t*)x.packed, (int)x.n / 16, (int)x.k / 32};
      const int64_t items = (x.n / 16) * (x.k / 32);
      most = items > most ? items : most;
    }
    a.n = count;
    a.gelu_table = first == 0 ? gelu_table : nullptr;
    const unsigned pack_blocks = (unsigned)((most + 3) / 4), parts = count + (a.gelu_table ? 1 : 0);
    bool joint = false;
    if (first == 0 && norm && norm->rows > 0) {
      const auto go = [&](auto type, auto lanes) {
        constexpr int LPR = decltype(lanes)::value, RPB = 256 / LPR;
        const NormArgs r = {(const uint16_t*)norm->x, (const uint16_t*)norm->weight, (const uint16_t*)norm->bias, (uint16_t*)norm->y, norm->eps,
                            (int)norm->rows, (int)norm->dim, (int)((norm->rows + RPB - 1) / RPB)};
        const int64_t nblk = pack_and_norm_blocks(norm->rows, RPB, pack_blocks, parts);
        if ((joint = nblk > 0))
          hipLaunchKernelGGL((pack_and_norm_kernel<decltype(type), LPR>), dim3((unsigned)nblk), dim3(256), 0, stream, a, r, (int)pack_blocks);
      };
      const auto by_width = [&](auto type) {  // as launch_layer_norm
        if (norm->dim <= 128) return go(type, std::integral_constant<int, 16>{});
        if (norm->dim <= 256) return go(type, std::integral_constant<int, 32>{});
        return go(type, std::integral_constant<int, 64>{});
      };
      norm->dtype == 0 ? by_width(BF16{}) : by_width(FP16{});
      if (!joint) {
        const hipError_t en = launch_layer_norm(norm->dtype, norm->rows, norm->dim, norm->x, norm->weight, norm->bias, norm->eps, norm->y, stream);
        if (en != hipSuccess) return en;
      }
    }
    if (!joint) hipLaunchKernelGGL(pack_weights_kernel, dim3(pack_blocks, parts), dim3(256), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_block_tail(const moda_hip_block_tail_args* t, int compute_units, hipStream_t stream) {
  const TailArgs a = tail_args(t);
  return t->dtype == 0 ? launch_tail<BF16>(a, (int)t->width, t->post_norm != 0, compute_units, stream)
                       : launch_tail<FP16>(a, (int)t->width, t->post_norm != 0, compute_units, stream);
}

}  // namespace moda
