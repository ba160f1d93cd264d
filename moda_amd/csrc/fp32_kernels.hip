// Exact fp32 attention on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32): forward, dQ and dK/dV of every mode
// for head dims up to 128 -- the computation of moda_v14.py:45-378, 542-1454, moda_v16.py and fda_v12.py with fp32
// operands, fp32 products and fp32 sums throughout.
//
// Shape of the work.  fp32 problems are small (gradient checks, fine-tuning of small models): a few hundred rows
// per head, so what counts is how many waves the problem is cut into and how short each wave's chain is.  A
// workgroup of W waves owns 16 query rows (forward, dQ) or 16 sequence keys (dK/dV); its waves take the 16-wide
// blocks of the other axis in turn, each with partial results of its own, and meet once, at the end, in LDS.  There
// is no barrier and no LDS traffic before that: operands go from global memory (L2 after first touch) straight into
// the registers the matrix instruction reads, one block ahead of their use.  At 32 cycles per instruction and SIMD
// a 16-wide block of head dim 128 keeps the matrix pipe busy for 2048 cycles per 16 KB fetched, which L2 can feed.
// A depth slot is seen by few rows (its token's, or its chunk's), so there a wave owns 16 slots by itself.
//
// Operand layout, lane l = (n, q), n = l & 15, q = l >> 4.  A (16 x 4): row n, summation slot q.  B (4 x 16): column n,
// slot q.  C: column n, rows 4q + i.  Summation slots are free to name:
//   scores (sum over the head dim): step (s, i) takes head-dim element 16 s + 4 q + i in slot q, so a lane's operand of
//     four steps is one 16-byte piece of its row;
//   second products (sum over the scores' rows): step i takes row 4 q + i in slot q, which is where the scores'
//     accumulators already are; the other operand is the 16-byte piece of row 4 q + i at element 64 h + 4 n, four
//     output blocks at once (block (h, j) holds head-dim element 64 h + 4 m + j on row m).
//
// B=1 T=256 H=4 D=64 L=4 causal, forward + backward: 336 us of kernels on the vector-ALU kernels of
// generic_kernels.hip (one wave per row or column, element loads), which remain for what is not covered here.
#include "geometry.h"
#include "kargs.h"
#include "tile.h"

namespace moda {

namespace {

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ float quad_sum_f32(float x) {  // over the four lanes that share n
  x += __shfl_xor(x, 16, 64);
  return pair_sum(x);
}
__device__ __forceinline__ float quad_max_f32(float x) {
  x = fmaxf(x, __shfl_xor(x, 16, 64));
  return pair_max(x);
}

// The lane's pieces of one row as a score operand: elements 16 s + 4 q .. +3.  FULL: the tensor's head dim is HD;
// otherwise pieces past the head dim `d` read the row's start and count as zero.
template <int HD, bool FULL>
__device__ __forceinline__ void load_score_operand(f32x4 (&x)[HD / 16], const float* row, int q, int d) {
#pragma unroll
  for (int s = 0; s < HD / 16; s++) {
    const bool in = FULL || 16 * s + 4 * q < d;
    const f32x4 v = *reinterpret_cast<const f32x4*>(row + (in ? 16 * s + 4 * q : 0));
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    x[s] = in ? v : z;
  }
}
// The lane's piece of row 4 q + i as the second products' operand: elements 64 h + 4 n .. +3.
template <int HD, bool FULL>
__device__ __forceinline__ void load_sum_operand(f32x4 (&x)[HD / 64], const float* row, int n, int d) {
#pragma unroll
  for (int h = 0; h < HD / 64; h++) {
    const bool in = FULL || 64 * h + 4 * n < d;
    const f32x4 v = *reinterpret_cast<const f32x4*>(row + (in ? 64 * h + 4 * n : 0));
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    x[h] = in ? v : z;
  }
}

// init + rows(x) . rows(y) over the head dim, two accumulators so that consecutive instructions are independent
template <int HD>
__device__ __forceinline__ f32x4 scores(const f32x4 (&x)[HD / 16], const f32x4 (&y)[HD / 16], f32x4 init) {
  f32x4 s0 = init, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < HD / 16; s++)
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      s0 = mfma_f32(x[s][i], y[s][i], s0);
      s1 = mfma_f32(x[s][i + 1], y[s][i + 1], s1);
    }
  return s0 + s1;
}

// acc[h][j] += (element 64 h + 4 m + j of rows 4 q + i) x w[i]
template <int HD>
__device__ __forceinline__ void accumulate(f32x4 (&acc)[HD / 64][4], const f32x4 (&x)[4][HD / 64], const f32x4& w) {
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int h = 0; h < HD / 64; h++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[h][j] = mfma_f32(x[i][h][j], w[i], acc[h][j]);
}

// The same where not every column sees every row (`see`: the lane's column sees row 4 q + i).  The weight of an unseen
// pair is zero, which takes a finite row out of the product but not one with an infinity or a NaN in it: 0 x those is
// NaN, and a later token's value would reach an earlier token's result.  A block that holds such a value is added up
// pair by pair, unseen pairs left out.  Finding out costs HD / 4 vector instructions beside HD / 4 matrix instructions
// of 32 cycles, in blocks on an edge of what is visible and in depth blocks only.
template <int HD>
__device__ __forceinline__ void accumulate_seen(f32x4 (&acc)[HD / 64][4], const f32x4 (&x)[4][HD / 64], const f32x4& w, const bool (&see)[4],
                                                int n, int q) {
  float z = 0.f;
  if (!__all(see[0] && see[1] && see[2] && see[3]))
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int h = 0; h < HD / 64; h++)
#pragma unroll
        for (int j = 0; j < 4; j++) z = __builtin_fmaf(x[i][h][j], 0.f, z);
  if (!__any(z != 0.f)) {  // NaN as soon as one of them is not finite
    accumulate<HD>(acc, x, w);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll 1
    for (int g = 0; g < 4; g++) {  // row 4 g + i; its element 64 h + 16 q + 4 m + j is with lane 4 q + m of the rows' group g
      const float weight = __shfl(w[i], 16 * g + n, 64);
      const bool seen = __shfl((int)see[i], 16 * g + n, 64) != 0;
#pragma unroll
      for (int h = 0; h < HD / 64; h++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
          for (int m = 0; m < 4; m++) {
            const float v = __shfl(x[i][h][j], 16 * g + 4 * q + m, 64);
            acc[h][j][m] = seen ? __builtin_fmaf(v, weight, acc[h][j][m]) : acc[h][j][m];
          }
          __builtin_amdgcn_sched_barrier(0);  // a few values at a time: the registers of this path are those of the kernel
        }
    }
}

template <int HD>
__device__ __forceinline__ void clear(f32x4 (&acc)[HD / 64][4]) {
#pragma unroll
  for (int h = 0; h < HD / 64; h++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[h][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}
// the four consecutive head-dim elements 64 h + 16 q + 4 i .. +3 of the lane's column
template <int HD>
__device__ __forceinline__ f32x4 piece(const f32x4 (&acc)[HD / 64][4], int h, int i) {
  return f32x4{acc[h][0][i], acc[h][1][i], acc[h][2][i], acc[h][3][i]};
}
// partial results of one wave in LDS: 16 rows, padded by one 16-byte piece against bank conflicts
template <int HD>
constexpr int kPartRow = HD + 4;
template <int HD>
__device__ __forceinline__ void leave_partial(float* part, const f32x4 (&acc)[HD / 64][4], int n, int q) {
#pragma unroll
  for (int h = 0; h < HD / 64; h++)
#pragma unroll
    for (int i = 0; i < 4; i++) *reinterpret_cast<f32x4*>(part + n * kPartRow<HD> + 64 * h + 16 * q + 4 * i) = piece<HD>(acc, h, i);
}

// What the row kernels' column block `blk` is: sequence keys, then the depth slots the 16 rows can see.
struct Block {
  const float *k, *v;  // (batch, head) slices
  int64_t sk, sv;      // row strides
  int col0, ncols;     // first column, columns of the axis
  bool dep;
};
__device__ __forceinline__ Block column_block(const KArgs& a, const RowTilePlan& plan, int blk, int b, int hkv) {
  Block x;
  x.dep = blk >= plan.n_seq;
  if (!x.dep) {
    x.k = (const float*)a.k + b * a.sk.b + hkv * a.sk.h;
    x.v = (const float*)a.v + b * a.sv.b + hkv * a.sv.h;
    x.sk = a.sk.t;
    x.sv = a.sv.t;
    x.col0 = blk * 16;
    x.ncols = a.T;
  } else {
    x.k = (const float*)a.kd + b * a.skd.b + hkv * a.skd.h;
    x.v = (const float*)a.vd + b * a.svd.b + hkv * a.svd.h;
    x.sk = a.skd.t;
    x.sv = a.svd.t;
    x.col0 = plan.dep0 + (blk - plan.n_seq) * 16;
    x.ncols = a.T * a.Lv;
  }
  return x;
}
// tensor row of column c (columns past the end read the last one; their scores are masked)
__device__ __forceinline__ int64_t block_row(const KArgs& a, const Block& x, int c) {
  c = imin(c, x.ncols - 1);
  return x.dep ? depth_row_of(a, c) : (int64_t)c;
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

}  // namespace

constexpr int kFp32RowWaves = 8;

template <int HD, bool FULL>
__global__ __launch_bounds__(64 * kFp32RowWaves, 2) void fp32_fwd_kernel(const KArgs a_in) {
  constexpr int W = kFp32RowWaves, KS = HD / 16, H4 = HD / 64;
  extern __shared__ __align__(16) float fp32_smem[];
  float* part = fp32_smem;                       // [W][16][HD + 4]
  float* ml = fp32_smem + W * 16 * kPartRow<HD>;  // [W][16][2]: exponent reference, row sum
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4, wave = uniform(tid >> 6);
  KArgs a = a_in;
  const int BH = a.B * a.Hq, bh = blockIdx.x % BH;
  int b = bh / a.Hq;
  const int hq = bh % a.Hq, hkv = hq / a.hdiv;
  enter_sequence(a, b, 2);
  const int qt = query_tile_of(blockIdx.x, BH, 16, a_in.Tq);
  if (qt * 16 >= a.Tq) return;  // a tile beyond this sequence of a packed batch
  const int r = qt * 16 + n, rc = imin(r, a.Tq - 1);
  f32x4 Q[KS];
  load_score_operand<HD, FULL>(Q, (const float*)a.q + b * a.sq.b + hq * a.sq.h + rc * a.sq.t, q, a.D);
  const RowVis vis = row_visibility(a, r, a.L);
  RowTilePlan plan = row_tile_plan(a, qt, 16, 16, a.L > 0);
  plan.n_seq = uniform(plan.n_seq);
  const int nblk = plan.n_seq + uniform(plan.n_dep);

  f32x4 o[H4][4];
  clear<HD>(o);
  float m = kNegInf, l = 0.f;
  const float sc = a.scale * kLog2e;
  f32x4 K[KS], V[4][H4];
  auto load_k = [&](int blk) {
    const Block x = column_block(a, plan, blk, b, hkv);
    load_score_operand<HD, FULL>(K, x.k + block_row(a, x, x.col0 + n) * x.sk, q, a.D);
  };
  if (wave < nblk) load_k(wave);
  for (int blk = wave; blk < nblk; blk += W) {
    const Block x = column_block(a, plan, blk, b, hkv);
#pragma unroll
    for (int i = 0; i < 4; i++) load_sum_operand<HD, FULL>(V[i], x.v + block_row(a, x, x.col0 + 4 * q + i) * x.sv, n, a.Dv);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 s = scores<HD>(K, Q, f32x4{0.f, 0.f, 0.f, 0.f});
    if (blk + W < nblk) load_k(blk + W);
    __builtin_amdgcn_sched_barrier(0);
    const int lo = x.dep ? vis.dlo : 0, hi = x.dep ? vis.dhi : vis.shi;
    float mx = kNegInf;
    bool see[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = x.col0 + 4 * q + i;
      see[i] = c >= lo && c < hi;
      s[i] = see[i] ? s[i] * sc : kNegInf;
      mx = fmaxf(mx, s[i]);
    }
    // the exponent reference only moves when a score outgrows it by more than 2^8 (exact in fp32 up to there)
    if (__any(mx > m + 8.f)) {
      const float m_new = fmaxf(m, quad_max_f32(mx));
      const float alpha = exp2f(m - ((m_new == kNegInf) ? 0.f : m_new));
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int h = 0; h < H4; h++)
#pragma unroll
        for (int j = 0; j < 4; j++) o[h][j] *= alpha;
    }
    const float ref = (m == kNegInf) ? 0.f : m;
    f32x4 p;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      p[i] = see[i] ? exp2f(s[i] - ref) : 0.f;
      l += p[i];
    }
    accumulate_seen<HD>(o, V, p, see, n, q);
  }
  l = quad_sum_f32(l);
  leave_partial<HD>(part + wave * 16 * kPartRow<HD>, o, n, q);
  if (q == 0) {
    ml[(wave * 16 + n) * 2] = m;
    ml[(wave * 16 + n) * 2 + 1] = l;
  }
  __syncthreads();
  // one thread per row and four head-dim elements
  const int row = tid / (HD / 4), d = (tid % (HD / 4)) * 4;
  if (tid < 16 * HD / 4 && qt * 16 + row < a.Tq) {
    const int nw = imin(W, nblk);
    float M = kNegInf;
    for (int w = 0; w < nw; w++) M = fmaxf(M, ml[(w * 16 + row) * 2]);
    const float ref = (M == kNegInf) ? 0.f : M;
    float L = 0.f;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < nw; w++) {
      const float f = exp2f(ml[(w * 16 + row) * 2] - ref);
      L += f * ml[(w * 16 + row) * 2 + 1];
      x += *reinterpret_cast<const f32x4*>(part + (w * 16 + row) * kPartRow<HD> + d) * f;
    }
    const int ro = qt * 16 + row;
    x *= L > 0.f ? 1.f / L : 0.f;
    if (d < a.Dv) *reinterpret_cast<f32x4*>((float*)a.out_o + b * a.so.b + hq * a.so.h + ro * a.so.t + d) = x;
    if (d == 0) a.lse[((int64_t)b * a.Tq + ro) * a.Hq + hq] = L > 0.f ? M + log2f(L) : kNegInf;
  }
}

// Minus rowsum(o * do) of one row from the lane's score-operand pieces of both, in all four lanes of the row.
template <int HD>
__device__ __forceinline__ float neg_delta_of(const f32x4 (&o)[HD / 16], const f32x4 (&d_o)[HD / 16]) {
  float acc = 0.f;
#pragma unroll
  for (int s = 0; s < HD / 16; s++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc = __builtin_fmaf(o[s][i], d_o[s][i], acc);
  return -quad_sum_f32(acc);
}

// `block`: this workgroup's place among the launch's dQ workgroups
template <int HD, bool FULL>
__device__ __forceinline__ void fp32_dq_body(const KArgs& a_in, int block) {
  constexpr int W = kFp32RowWaves, KS = HD / 16, H4 = HD / 64;
  extern __shared__ __align__(16) float fp32_smem[];
  float* part = fp32_smem;  // [W][16][HD + 4]
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4, wave = uniform(tid >> 6);
  KArgs a = a_in;
  const int BH = a.B * a.Hq, bh = block % BH;
  int b = bh / a.Hq;
  const int hq = bh % a.Hq, hkv = hq / a.hdiv;
  enter_sequence(a, b, 2);
  const int qt = query_tile_of(block, BH, 16, a_in.Tq);
  if (qt * 16 >= a.Tq) return;
  const int r = qt * 16 + n, rc = imin(r, a.Tq - 1);
  f32x4 Q[KS], dO[KS];
  load_score_operand<HD, FULL>(Q, (const float*)a.q + b * a.sq.b + hq * a.sq.h + rc * a.sq.t, q, a.D);
  load_score_operand<HD, FULL>(dO, (const float*)a.d_o + b * a.sdo.b + hq * a.sdo.h + rc * a.sdo.t, q, a.Dv);
  float neg_delta;
  {
    f32x4 O[KS];
    load_score_operand<HD, FULL>(O, (const float*)a.o + b * a.so.b + hq * a.so.h + rc * a.so.t, q, a.Dv);
    neg_delta = neg_delta_of<HD>(O, dO);
  }
  const float lse = a.lse[((int64_t)b * a.Tq + rc) * a.Hq + hq];
  if (wave == 0 && q == 0 && r < a.Tq) a.delta[((int64_t)b * a.Hq + hq) * a.delta_pitch + r] = neg_delta;
  const RowVis vis = row_visibility(a, r, a.L);
  RowTilePlan plan = row_tile_plan(a, qt, 16, 16, a.L > 0);
  plan.n_seq = uniform(plan.n_seq);
  const int nblk = plan.n_seq + uniform(plan.n_dep);

  f32x4 dq[H4][4];
  clear<HD>(dq);
  const float sc = a.scale * kLog2e;
  f32x4 K[KS], V[KS], KT[4][H4];
  auto load_kv = [&](int blk) {
    const Block x = column_block(a, plan, blk, b, hkv);
    const int64_t row = block_row(a, x, x.col0 + n);
    load_score_operand<HD, FULL>(K, x.k + row * x.sk, q, a.D);
    load_score_operand<HD, FULL>(V, x.v + row * x.sv, q, a.Dv);
  };
  if (wave < nblk) load_kv(wave);
  for (int blk = wave; blk < nblk; blk += W) {
    const Block x = column_block(a, plan, blk, b, hkv);
#pragma unroll
    for (int i = 0; i < 4; i++) load_sum_operand<HD, FULL>(KT[i], x.k + block_row(a, x, x.col0 + 4 * q + i) * x.sk, n, a.D);
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 s = scores<HD>(K, Q, f32x4{0.f, 0.f, 0.f, 0.f});
    const f32x4 dp = scores<HD>(V, dO, f32x4{neg_delta, neg_delta, neg_delta, neg_delta});
    if (blk + W < nblk) load_kv(blk + W);
    __builtin_amdgcn_sched_barrier(0);
    const int lo = x.dep ? vis.dlo : 0, hi = x.dep ? vis.dhi : vis.shi;
    f32x4 ds;
    bool see[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = x.col0 + 4 * q + i;
      see[i] = c >= lo && c < hi;
      ds[i] = see[i] ? exp2f(__builtin_fmaf(s[i], sc, -lse)) * dp[i] : 0.f;
    }
    accumulate_seen<HD>(dq, KT, ds, see, n, q);
  }
  leave_partial<HD>(part + wave * 16 * kPartRow<HD>, dq, n, q);
  __syncthreads();
  const int row = tid / (HD / 4), d = (tid % (HD / 4)) * 4;
  if (tid < 16 * HD / 4 && qt * 16 + row < a.Tq && d < a.D) {
    const int nw = imin(W, nblk);
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < nw; w++) x += *reinterpret_cast<const f32x4*>(part + (w * 16 + row) * kPartRow<HD> + d);
    *reinterpret_cast<f32x4*>((float*)a.dq + b * a.sdq.b + hq * a.sdq.h + (qt * 16 + row) * a.sdq.t + d) = x * a.scale;
  }
}

template <int HD, bool FULL>
__global__ __launch_bounds__(64 * kFp32RowWaves, 2) void fp32_dq_kernel(const KArgs a) {
  fp32_dq_body<HD, FULL>(a, blockIdx.x);
}

// Minus rowsum(o * do) alone, for a dK/dV stage that runs without the dQ stage: one wave per 16 rows.
template <int HD, bool FULL>
__global__ __launch_bounds__(64) void fp32_delta_kernel(const KArgs a_in) {
  const int lane = threadIdx.x, n = lane & 15, q = lane >> 4;
  KArgs a = a_in;
  const int BH = a.B * a.Hq, bh = blockIdx.x % BH;
  int b = bh / a.Hq;
  const int hq = bh % a.Hq;
  enter_sequence(a, b, 2);
  const int r = (blockIdx.x / BH) * 16 + n, rc = imin(r, a.Tq - 1);
  if (rc < 0) return;  // an empty sequence of a packed batch
  f32x4 O[HD / 16], dO[HD / 16];
  load_score_operand<HD, FULL>(O, (const float*)a.o + b * a.so.b + hq * a.so.h + rc * a.so.t, q, a.Dv);
  load_score_operand<HD, FULL>(dO, (const float*)a.d_o + b * a.sdo.b + hq * a.sdo.h + rc * a.sdo.t, q, a.Dv);
  const float x = neg_delta_of<HD>(O, dO);
  if (q == 0 && r < a.Tq) a.delta[((int64_t)b * a.Hq + hq) * a.delta_pitch + r] = x;
}

// dK/dV.  The grid holds, per (batch, kv head), the 16-key tiles of the sequence (a workgroup each, its waves share the
// query rows), then workgroups of W times 16 depth slots (a wave each).  At head dim 128 four waves with the whole
// register file rather than eight with half of it: stationary rows, accumulators and both forms of a query block
// together take more than 256 registers.
template <int HD>
constexpr int kFp32ColWaves = HD <= 64 ? 8 : 4;

// `block`: this workgroup's place among the launch's dK/dV workgroups.  OWN_DELTA: the row sums of o * do are formed here, block
// by block (a launch that runs beside the dQ workgroups cannot read theirs); the same additions in the same order as there
template <int HD, bool FULL, bool OWN_DELTA>
__device__ __forceinline__ void fp32_dkv_body(const KArgs& a_in, int block) {
  constexpr int W = kFp32ColWaves<HD>, KS = HD / 16, H4 = HD / 64, PART = 16 * kPartRow<HD>;
  extern __shared__ __align__(16) float fp32_smem[];
  float* part = fp32_smem;  // [2 (dk, dv)][W][16][HD + 4]
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4, wave = uniform(tid >> 6);
  KArgs a = a_in;
  const int BHk = a.B * a.Hkv, bh = block % BHk;
  int b = bh / a.Hkv;
  const int hkv = bh % a.Hkv, tile = block / BHk, n_seq_tiles = a_in.has_seq ? (a_in.T + 15) / 16 : 0;
  enter_sequence(a, b, 2);
  const bool dep = tile >= n_seq_tiles;
  const int ncols = dep ? a.T * a.Lv : a.T;
  const int c0 = dep ? ((tile - n_seq_tiles) * W + wave) * 16 : tile * 16;
  if (c0 >= ncols) return;  // the whole workgroup for a sequence tile, single waves (which meet no barrier) for slots
  const int c = c0 + n;
  const bool valid = c < ncols;
  const int cc = imin(c, ncols - 1);
  const int64_t crow = dep ? depth_row_of(a, cc) : (int64_t)cc;
  f32x4 K[KS], V[KS];
  load_score_operand<HD, FULL>(K, dep ? (const float*)a.kd + b * a.skd.b + hkv * a.skd.h + crow * a.skd.t
                                      : (const float*)a.k + b * a.sk.b + hkv * a.sk.h + crow * a.sk.t, q, a.D);
  load_score_operand<HD, FULL>(V, dep ? (const float*)a.vd + b * a.svd.b + hkv * a.svd.h + crow * a.svd.t
                                      : (const float*)a.v + b * a.sv.b + hkv * a.sv.h + crow * a.sv.t, q, a.Dv);
  int qlo = 0, qhi = 0, wg_lo, wg_hi, unused;
  if (valid) q_interval(a, dep, c, qlo, qhi);
  q_interval(a, dep, c0, wg_lo, unused);
  q_interval(a, dep, imin(ncols, c0 + 16) - 1, unused, wg_hi);
  const int r_first = uniform(wg_lo) / 16 * 16, nrb = (uniform(wg_hi) - r_first + 15) / 16;  // row blocks of a query head
  const int nblk = nrb * a.hdiv;  // hdiv > 1: head-dim GQA, the query heads of this kv head one after the other

  f32x4 dk[H4][4], dv[H4][4];
  clear<HD>(dk);
  clear<HD>(dv);
  const float sc = a.scale * kLog2e;
  f32x4 Q[KS], dO[KS], QT[4][H4], dOT[4][H4];
  f32x4 O[OWN_DELTA ? KS : 1];
  float lse[4], neg_delta[4];
  struct Rows {
    const float *q, *d_o;  // slices of the query head
    int hq, r0;
  };
  auto rows_of = [&](int blk) {
    const int gh = blk / nrb, hq = hkv * a.hdiv + gh;
    return Rows{(const float*)a.q + b * a.sq.b + hq * a.sq.h, (const float*)a.d_o + b * a.sdo.b + hq * a.sdo.h, hq,
                r_first + (blk - gh * nrb) * 16};
  };
  auto load_rows = [&](int blk) {
    const Rows x = rows_of(blk);
    const int64_t r = imin(x.r0 + n, a.Tq - 1);
    load_score_operand<HD, FULL>(Q, x.q + r * a.sq.t, q, a.D);
    load_score_operand<HD, FULL>(dO, x.d_o + r * a.sdo.t, q, a.Dv);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int ri = imin(x.r0 + 4 * q + i, a.Tq - 1);
      lse[i] = a.lse[((int64_t)b * a.Tq + ri) * a.Hq + x.hq];
      if (!OWN_DELTA) neg_delta[i] = a.delta[((int64_t)b * a.Hq + x.hq) * a.delta_pitch + ri];
    }
    if constexpr (OWN_DELTA) load_score_operand<HD, FULL>(O, (const float*)a.o + b * a.so.b + x.hq * a.so.h + r * a.so.t, q, a.Dv);
  };
  const int blk0 = dep ? 0 : wave, step = dep ? 1 : W;
  if (blk0 < nblk) load_rows(blk0);
  for (int blk = blk0; blk < nblk; blk += step) {
    const Rows x = rows_of(blk);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int64_t r = imin(x.r0 + 4 * q + i, a.Tq - 1);
      load_sum_operand<HD, FULL>(QT[i], x.q + r * a.sq.t, n, a.D);
      load_sum_operand<HD, FULL>(dOT[i], x.d_o + r * a.sdo.t, n, a.Dv);
    }
    if constexpr (OWN_DELTA) {  // lane (n, .) has the sum of row n, its accumulators hold rows 4 q + i
      const float row_sum = neg_delta_of<HD>(O, dO);
#pragma unroll
      for (int i = 0; i < 4; i++) neg_delta[i] = __shfl(row_sum, 4 * q + i, 64);
    }
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 s = scores<HD>(Q, K, f32x4{0.f, 0.f, 0.f, 0.f});
    const f32x4 dp = scores<HD>(dO, V, f32x4{neg_delta[0], neg_delta[1], neg_delta[2], neg_delta[3]});
    f32x4 p, ds;
    bool see[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = x.r0 + 4 * q + i;
      see[i] = r >= qlo && r < qhi;
      p[i] = see[i] ? exp2f(__builtin_fmaf(s[i], sc, -lse[i])) : 0.f;
      ds[i] = see[i] ? p[i] * dp[i] : 0.f;
    }
    if (blk + step < nblk) load_rows(blk + step);
    __builtin_amdgcn_sched_barrier(0);
    accumulate_seen<HD>(dv, dOT, p, see, n, q);
    accumulate_seen<HD>(dk, QT, ds, see, n, q);
  }

  if (dep) {
    if (!valid) return;
    float* dkp = (float*)a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + crow * a.sdkd.t;
    float* dvp = (float*)a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + crow * a.sdvd.t;
#pragma unroll
    for (int h = 0; h < H4; h++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int d = 64 * h + 16 * q + 4 * i;
        f32x4 x = piece<HD>(dk, h, i) * a.scale, y = piece<HD>(dv, h, i);
        if (a.accum_depth) {  // add to what the row holds (this lane is its only writer)
          if (d < a.D) x += *reinterpret_cast<f32x4*>(dkp + d);
          if (d < a.Dv) y += *reinterpret_cast<f32x4*>(dvp + d);
        }
        if (d < a.D) *reinterpret_cast<f32x4*>(dkp + d) = x;
        if (d < a.Dv) *reinterpret_cast<f32x4*>(dvp + d) = y;
      }
    // the lane group of a token's last filled slot also clears the rows of the slots without data
    if (a.Lv != a.L && !a.keep_slots && c % a.Lv == a.Lv - 1) {
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      for (int slot = a.Lv; slot < a.L; slot++) {
        dkp += a.sdkd.t;
        dvp += a.sdvd.t;
        for (int d = 4 * q; d < a.D; d += 16) *reinterpret_cast<f32x4*>(dkp + d) = z;
        for (int d = 4 * q; d < a.Dv; d += 16) *reinterpret_cast<f32x4*>(dvp + d) = z;
      }
    }
    return;
  }
  leave_partial<HD>(part + wave * PART, dk, n, q);
  leave_partial<HD>(part + (W + wave) * PART, dv, n, q);
  __syncthreads();
  const int nw = imin(W, nblk);
  for (int e = tid; e < 2 * 16 * HD / 4; e += 64 * W) {
    const int which = e / (16 * HD / 4), row = e % (16 * HD / 4) / (HD / 4), d = (e % (HD / 4)) * 4;
    if (c0 + row >= ncols || d >= (which ? a.Dv : a.D)) continue;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < nw; w++) x += *reinterpret_cast<const f32x4*>(part + (which * W + w) * PART + row * kPartRow<HD> + d);
    if (which)
      *reinterpret_cast<f32x4*>((float*)a.dv + b * a.sdv.b + hkv * a.sdv.h + (int64_t)(c0 + row) * a.sdv.t + d) = x;
    else
      *reinterpret_cast<f32x4*>((float*)a.dk + b * a.sdk.b + hkv * a.sdk.h + (int64_t)(c0 + row) * a.sdk.t + d) = x * a.scale;
  }
}

template <int HD, bool FULL>
__global__ __launch_bounds__(64 * kFp32ColWaves<HD>, HD <= 64 ? 2 : 1) void fp32_dkv_kernel(const KArgs a) {
  fp32_dkv_body<HD, FULL, false>(a, blockIdx.x);
}

// dQ and dK/dV of a problem that leaves compute units idle in one launch, their workgroups side by side: two chains of a few
// dependent blocks behind one start and one end.  B=1 T=256 H=4 D=64 L=4 causal: the replayed training step 33.1 -> 23.9 us.
template <bool FULL>
__global__ __launch_bounds__(64 * kFp32RowWaves, 2) void fp32_bwd_kernel(const KArgs a, int row_blocks) {
  static_assert(kFp32ColWaves<64> == kFp32RowWaves, "workgroups of one size");
  if ((int)blockIdx.x < row_blocks)
    fp32_dq_body<64, FULL>(a, blockIdx.x);
  else
    fp32_dkv_body<64, FULL, true>(a, (int)blockIdx.x - row_blocks);
}

namespace {

template <typename Kernel, typename... More>
hipError_t launch(Kernel kernel, LdsAttrState& attr, const KArgs& a, int64_t nblk, int threads, size_t smem, hipStream_t stream, More... more) {
  if (nblk == 0) return hipSuccess;
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  const hipError_t e = allow_dynamic_lds(attr, reinterpret_cast<const void*>(kernel), smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)nblk), dim3(threads), smem, stream, a, more...);
  return hipGetLastError();
}

template <int HD, bool FULL>
hipError_t launch_fp32_t(const KArgs& a, int which, hipStream_t stream) {
  constexpr size_t part = (size_t)16 * kPartRow<HD> * sizeof(float);
  static LdsAttrState attr[5];
  const int64_t row_tiles = (int64_t)((a.Tq + 15) / 16) * a.B * a.Hq;
  if (which == 0)
    return launch(&fp32_fwd_kernel<HD, FULL>, attr[0], a, row_tiles, 64 * kFp32RowWaves,
                  kFp32RowWaves * (part + 32 * sizeof(float)), stream);
  if (which == 1) return launch(&fp32_dq_kernel<HD, FULL>, attr[1], a, row_tiles, 64 * kFp32RowWaves, kFp32RowWaves * part, stream);
  if (which == 3) return launch(&fp32_delta_kernel<HD, FULL>, attr[3], a, row_tiles, 64, 0, stream);
  constexpr int W = kFp32ColWaves<HD>;
  const int64_t seq = a.has_seq ? (a.T + 15) / 16 : 0, dep = ((int64_t)a.T * a.Lv + 16 * W - 1) / (16 * W);
  const int64_t columns = (seq + dep) * a.B * a.Hkv;
  if constexpr (HD == 64) {
    if (which == 4) return launch(&fp32_bwd_kernel<FULL>, attr[4], a, row_tiles + columns, 64 * W, 2 * W * part, stream, (int)row_tiles);
  }
  return launch(&fp32_dkv_kernel<HD, FULL>, attr[2], a, columns, 64 * W, 2 * W * part, stream);
}

}  // namespace

// which: 4 dQ and dK/dV in one launch; 0 forward, 1 dQ (leaves the row sums of o * do in the workspace), 2 dK/dV (reads them), 3 the row sums alone
hipError_t launch_fp32(const KArgs& a, int which, hipStream_t stream) {
  const int hd = a.D > a.Dv ? a.D : a.Dv;
  if (hd <= 64) return a.D == 64 && a.Dv == 64 ? launch_fp32_t<64, true>(a, which, stream) : launch_fp32_t<64, false>(a, which, stream);
  if (hd <= 128) return a.D == 128 && a.Dv == 128 ? launch_fp32_t<128, true>(a, which, stream) : launch_fp32_t<128, false>(a, which, stream);
  return hipErrorInvalidValue;
}

}  // namespace moda
