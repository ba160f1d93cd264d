// The dense part of a transformer block in one launch: the body (block_tail_kernel.hip has what it computes and what bounds it).
#pragma once
#include <type_traits>

#include "../../include/moda_hip.h"
#include "block.h"
#ifdef MODA_SIDE_BY_SIDE
#include "fwd.h"
#endif
#include "tile.h"
#include "tile16.h"
#include "tuning.h"

namespace moda {

struct TailPart {
  const uint16_t *w, *bias;
  uint16_t* y;
  int64_t ldy;
  int block_end;  // 16-feature blocks of this part and of those before it
};
struct TailArgs {
  const uint16_t *h, *res;  // attention output, residual stream
  uint16_t* x;              // residual stream after the block
  int rows, hidden, n_parts;
  const uint16_t *proj_w, *proj_b, *fc1_w, *fc1_b, *fc2_w, *fc2_b;
  // layer norms: after the projection, and after the MLP (before-norm blocks: the next block's first norm)
  const uint16_t *mid_w, *mid_b, *end_w, *end_b;
  float mid_eps, end_eps;
  const float* gelu_table;  // bf16: written with the packed weights
  TailPart part[3];  // projections of the next block
};

namespace {

#define MODA_INLINE __attribute__((always_inline))  // lambdas: what they capture stays in registers

// workgroup barrier that waits for this wave's LDS accesses only: weights on their way to registers stay on their way
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// GELU of a packed pair of 16-bit values.  A bf16 value has 2 x 2688 magnitudes between 2^-17 and 16, outside of which the
// formula's result is x / 2 (to 6e-6, which no rounding to 8 bits sees), or 0 and x.  Inside, a table in LDS holds the formula's
// result, rounded, over x: times x that is the result again to 2^-23, which rounds to itself.  8 vector instructions an element
// where the formula (which fp16 takes) has 22, 6.5 k cycles for 64 rows x 256 features against 2.4 k (the launch 40 -> 32.7 us,
// before its sums took the order of the pieces).
constexpr int kGeluHalf = 21 * 128, kGeluTable = 2 * kGeluHalf, kGeluFirst = (127 - 17) << 7;
static_assert(kGeluTable * sizeof(float) == MODA_HIP_GELU_TABLE_BYTES, "what a caller allocates");
template <typename T>
constexpr int table_bytes() {
  return std::is_same<T, BF16>::value ? kGeluTable * 4 : 0;
}
template <typename T>
__device__ __forceinline__ int activated(int w, MODA_LDS const char* table) {
  float x[2];
  unpack2<T>(w, x[0], x[1]);
  if constexpr (table_bytes<T>() > 0) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    const u16x2 first = {kGeluFirst, kGeluFirst}, last = {kGeluHalf - 1, kGeluHalf - 1}, other = {4 * kGeluHalf, 4 * kGeluHalf};
    const u16x2 mag = __builtin_bit_cast(u16x2, w & 0x7fff7fff), sign = __builtin_bit_cast(u16x2, (int)(((unsigned)w >> 15) & 0x10001u));
    const u16x2 at = __builtin_elementwise_min(__builtin_elementwise_sub_sat(mag, first), last) * (unsigned short)4 + sign * other;
    const unsigned bytes = __builtin_bit_cast(unsigned, at);
    x[0] *= *reinterpret_cast<MODA_LDS const float*>(table + (bytes & 0xffffu));
    x[1] *= *reinterpret_cast<MODA_LDS const float*>(table + (bytes >> 16));
    return pack2<T>(x[0], x[1]);
  } else {
    return pack2<T>(gelu(x[0]), gelu(x[1]));
  }
}

// Sum of a row over the TPR neighbouring lanes (8 or 16) that share it; s[j] is what this lane has of the row's piece
// lsub + TPR j.  Added as layer_norm_kernel adds them, the two halves of the pieces first (past the last piece: zero).
template <int TPR, int NL>
__device__ __forceinline__ float row_sum(const float (&s)[NL]) {
  static_assert((TPR == 8 || TPR == 16) && NL <= 8, "half or whole rows of sixteen lanes");
  constexpr int P = NL > 4 ? 8 : NL > 2 ? 4 : NL;
  float t[P], v = 0.f;
#pragma unroll
  for (int j = 0; j < P; j++) t[j] = j < NL ? s[j] : 0.f;
#pragma unroll
  for (int h = P / 2; h > 0; h >>= 1)
#pragma unroll
    for (int j = 0; j < h; j++) t[j] += t[j + h];
  v = t[0];
#if defined(__HIP_DEVICE_COMPILE__)
  auto add = [&](auto ctrl) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  if (TPR == 16) add(std::integral_constant<int, 0x128>{});  // row_ror 8: the lane 8 away
  const int own = __builtin_bit_cast(int, v);  // the lane 4 away: row_shl 4 for banks 0 and 2, row_shr 4 for 1 and 3
  const int up = __builtin_amdgcn_update_dpp(0, own, 0x104, 0xf, 0x5, false);
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, own, 0x114, 0xf, 0xa, false));
  add(std::integral_constant<int, 0x4E>{});  // quad_perm 2, 3, 0, 1
  add(std::integral_constant<int, 0xB1>{});  // quad_perm 1, 0, 3, 2
#endif
  return v;
}

template <int W>
struct Rows : RowLayout<W> {
  // B operand of rows row0 + sigma(0..15), features 32 ks .. +31 (see Operand16); base: off(sigma(n), q4 + 4 j) for j = 0..3
  __device__ __forceinline__ static i32x4 operand(lds_cptr tile, const int (&base)[4], int row0, int ks) {
    return *reinterpret_cast<MODA_LDS const i32x4*>(tile + base[ks & 3] + row0 * W + (ks >> 2) * 128);
  }
};

// acc[mb][nb] += weights (MB blocks of 16 features) x rows (NB blocks of 16), K innermost.  PF steps of 32 of the weights
// are on their way; start() sends for the first ones, before what produces the rows.
template <typename T, int MB, int NB>
struct Product {
  static constexpr int PF = MB <= 3 ? 4 : 2;
  i32x4 w[PF][MB];
  const uint16_t* base[MB];  // wave-uniform: packed block of the features, at the first step of the sum
  uint32_t voff;             // this lane's byte offset

  __device__ __forceinline__ i32x4 get(int mb, int ks) const {
    typedef __attribute__((address_space(1))) const i32x4* vec;
    return *(vec)((__attribute__((address_space(1))) const char*)base[mb] + (size_t)voff + (size_t)ks * 1024);
  }
  __device__ __forceinline__ void load(int j) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++) w[j % PF][mb] = get(mb, j);
  }
  __device__ __forceinline__ void start() {
#pragma unroll
    for (int j = 0; j < PF; j++) load(j);
  }
  template <int W>
  __device__ __forceinline__ static void rows(i32x4 (&x)[NB], lds_cptr tile, const int (&rbase)[4], int ks) {
#pragma unroll
    for (int nb = 0; nb < NB; nb++) x[nb] = Rows<W>::operand(tile, rbase, 16 * nb, ks);
  }
  __device__ __forceinline__ void step(const i32x4 (&wj)[MB], const i32x4 (&x)[NB], f32x4 (&acc)[MB][NB]) const {
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++) acc[mb][nb] = mfma16<T>(wj[mb], x[nb], acc[mb][nb]);
  }
  // nk: steps of 32, a multiple of four.  The rows' operands of the next step are on their way while this one's products run.
  template <int W>
  __device__ __forceinline__ void run(lds_cptr tile, const int (&rbase)[4], int nk, f32x4 (&acc)[MB][NB]) {
    i32x4 x[2][NB];
    rows<W>(x[0], tile, rbase, 0);
    for (int k0 = 0; k0 < nk; k0 += 4) {
      lds_cptr at = tile + k0 * 32;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (j < 3 || k0 + 4 < nk) rows<W>(x[(j + 1) & 1], at, rbase, j + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(w[j % PF], x[j & 1], acc);
        if (k0 + j + PF < nk) {
#pragma unroll
          for (int mb = 0; mb < MB; mb++) w[j % PF][mb] = get(mb, k0 + j + PF);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // NK steps, all unrolled; after step j beside(j): work of another kind, or the loads of the product that follows
  template <int W, int NK, typename Beside>
  __device__ __forceinline__ void run_beside(lds_cptr tile, const int (&rbase)[4], f32x4 (&acc)[MB][NB], Beside&& beside) {
    i32x4 x[2][NB];
    rows<W>(x[0], tile, rbase, 0);
#pragma unroll
    for (int j = 0; j < NK; j++) {
      if (j + 1 < NK) rows<W>(x[(j + 1) & 1], tile, rbase, j + 1);
      __builtin_amdgcn_sched_barrier(0);
      step(w[j % PF], x[j & 1], acc);
      if (j + PF < NK) load(j + PF);
      __builtin_amdgcn_sched_barrier(0);
      beside(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

}  // namespace

// The same body with the block's attention before it (MODA_SIDE_BY_SIDE, attend_tail_kernel.hip): the workgroup forms the rows of H
// itself, from the arguments `att` of the forward kernel (fwd.h).  Its rows are then BM tokens of one sequence.
#ifdef MODA_SIDE_BY_SIDE
template <typename T, int C, int NB, bool POST, int ADDR, int KV_HEADS>
__global__ __launch_bounds__(512, 2) void attend_tail_kernel(const TailArgs a, const KArgs att) {
#else
template <typename T, int C, int NB, bool POST>
__global__ __launch_bounds__(512, 2) void block_tail_kernel(const TailArgs a) {
#endif
  constexpr int BM = 16 * NB, MB2 = C / 128, MB1 = 2, HC = 128 * MB1, CH = C / 8, TPR = 512 / BM, NL = CH / TPR;
  // The activation of a chunk beside the second product of the one before.  At width 256 that takes 15 to 31 registers more: with 32 rows
  // and POST room for two waves a SIMD instead of three (a workgroup has two, a second one never fitted), with 64 rows of bf16 five of
  // them spilled.  fp16's formula with 64 rows spills 23 (twelve blocks of width 256: 616 us apart, 624 beside), widths above 256 spill
  // more than they do apart.
  constexpr bool BESIDE = MB2 <= 2 && (NB == 2 || std::is_same<T, BF16>::value);
  static_assert(CH % TPR == 0, "a row's chunks over the threads of the row");
  extern __shared__ __align__(16) unsigned char tail_smem[];
  MODA_LDS const char* table = (MODA_LDS const char*)(lds_ptr)tail_smem;  // kGeluTable floats (bf16)
  lds_ptr X = (lds_ptr)tail_smem + (table_bytes<T>() / 2);  // [BM][C]: the block's rows
  lds_ptr H = X + BM * C;          // [BM][C] attention output, then two stages of [BM][HC] hidden activations
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#ifdef MODA_SIDE_BY_SIDE
  const AttendTailPlace at = attend_tail_place(att, blockIdx.x, BM);
  const int r0 = at.first_row, rows_end = at.rows_end;
#else
  const int r0 = blockIdx.x * BM, rows_end = a.rows;
#endif
  const int sigma = slot_base(n >> 2) + (n & 3);  // tile row of a 16-row block that lane column n stands for
  int xbase[4], hbase[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    xbase[j] = Rows<C>::off(sigma, 4 * j + q4);
    hbase[j] = Rows<HC>::off(sigma, 4 * j + q4);
  }
  const i32x2 none = {0, 0};
  auto unpack4 = [](const i32x2& w, float (&f)[4]) {
    unpack2<T>(w[0], f[0], f[1]);
    unpack2<T>(w[1], f[2], f[3]);
  };
  auto pack4 = [](const float (&f)[4]) {
    i32x2 w;
    w[0] = pack2<T>(f[0], f[1]);
    w[1] = pack2<T>(f[2], f[3]);
    return w;
  };
  auto zero = [](auto& acc) {
    for (auto& row : acc)
      for (auto& x : row) x = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  const int f2 = wave * 16 * MB2;  // this wave's features of a C-wide product
  // a bias's pieces at feature f of this wave, four features a lane
  auto pieces = [&](const uint16_t* bias, int f, auto& to) MODA_INLINE {
#pragma unroll
    for (int mb = 0; mb < (int)(sizeof(to) / sizeof(to[0])); mb++)
      to[mb] = bias ? *reinterpret_cast<const i32x2*>(bias + f + 16 * mb + 4 * q4) : none;
  };

  // Attention output, projection weights, residual and GELU table set out together, by rows (a load in the products' layout
  // would touch sixteen rows in each quarter of its lanes).
  Product<T, MB2, NB> proj;
  proj.voff = lane * 16;
  i32x2 bias2[MB2];
  {
    constexpr int N = BM * CH / 512, NT = table_bytes<T>() / 16;
    static_assert(BM * CH % 512 == 0, "whole passes");
    [[maybe_unused]] i32x4 v[N];
    i32x4 res[N], tab[(NT + 511) / 512 + 1];
    auto fetch = [&](const uint16_t* from, i32x4 (&to)[N]) MODA_INLINE {  // past the last row: that row's again, never stored
#pragma unroll
      for (int j = 0; j < N; j++) {
        const int row = r0 + (tid + 512 * j) / CH;
        to[j] = *reinterpret_cast<const i32x4*>(from + (int64_t)(row < rows_end ? row : rows_end - 1) * C + (tid + 512 * j) % CH * 8);
      }
    };
    auto leave = [&](lds_ptr tile, const i32x4 (&from)[N]) MODA_INLINE {
#pragma unroll
      for (int j = 0; j < N; j++) *reinterpret_cast<MODA_LDS i32x4*>(tile + Rows<C>::off((tid + 512 * j) / CH, (tid + 512 * j) % CH)) = from[j];
    };
#ifdef MODA_SIDE_BY_SIDE
    // residual and table travel with what the attention sends for first, and wait for it in registers
    fetch(a.res, res);
#pragma unroll
    for (int j = 0; j < (NT + 511) / 512; j++) tab[j] = reinterpret_cast<const i32x4*>(a.gelu_table)[tid + 512 * j < NT ? tid + 512 * j : 0];
    constexpr int G = C / 64 / KV_HEADS, WORK = BM * G / 32;
    typedef RowBlock<KV_HEADS, WORK> Shape;
    const int head = KV_HEADS > 1 ? wave / Shape::W : 0;
    fwd_body<T, 64, Shape, ADDR>(att, RowPlace{at.b, head, at.tile, 0, 0, true}, H + head * (Shape::NST * 2 * 64 * 64), X + head * (WORK * 32 * 64),
                                 H + attend_ring<Shape, BM>() + head * (WORK * 32 * 64), [&](int row, int chunk, int half, const i32x2& w) MODA_INLINE {
      *reinterpret_cast<MODA_LDS i32x2*>(H + Rows<C>::off(row / G, (row % G * KV_HEADS + head) * 8 + chunk) + 4 * half) = w;
    });
#pragma unroll
    for (int mb = 0; mb < MB2; mb++) proj.base[mb] = a.proj_w + (size_t)(f2 + 16 * mb) * C;
    proj.start();
    pieces(a.proj_b, f2, bias2);
    leave(X, res);
#else
    fetch(a.h, v);
#pragma unroll
    for (int mb = 0; mb < MB2; mb++) proj.base[mb] = a.proj_w + (size_t)(f2 + 16 * mb) * C;
    proj.start();
    fetch(a.res, res);
#pragma unroll
    for (int j = 0; j < (NT + 511) / 512; j++) tab[j] = reinterpret_cast<const i32x4*>(a.gelu_table)[tid + 512 * j < NT ? tid + 512 * j : 0];
    pieces(a.proj_b, f2, bias2);
    leave(H, v);
    leave(X, res);
#endif
#pragma unroll
    for (int j = 0; j < (NT + 511) / 512; j++)
      if (tid + 512 * j < NT) reinterpret_cast<MODA_LDS i32x4*>((lds_ptr)tail_smem)[tid + 512 * j] = tab[j];
  }
  i32x2 keep[MB2][NB];  // this lane's pieces of what the MLP's result is added to, rounded
  lds_barrier();
  f32x4 acc[MB2][NB];
  // (rows 16 apart share their swizzle: one address per feature block)
  auto own_piece = [&](int mb, int nb) { return X + Rows<C>::off(sigma, (f2 >> 3) + 2 * mb + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * C; };
  // + bias, rounded as the linear layer's result, + keep, rounded: into keep and the row tile
  auto add_keep = [&]() MODA_INLINE {
#pragma unroll
    for (int mb = 0; mb < MB2; mb++) {
      float b[4];
      unpack4(bias2[mb], b);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        float x[4], k[4];
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = acc[mb][nb][i] + b[i];
        unpack4(pack4(x), x);
        unpack4(keep[mb][nb], k);
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] += k[i];
        keep[mb][nb] = pack4(x);
        *reinterpret_cast<MODA_LDS i32x2*>(own_piece(mb, nb)) = keep[mb][nb];
      }
    }
  };
  // Layer norm of the row tile in place, TPR threads a row; `out`: the rows also go there, normalised (POST) or as they
  // were.  Parameters are fetched ahead of the barrier, by fetch_norm.
  const int lrow = tid / TPR, lsub = tid % TPR;
  i32x4 wv[NL], bv[NL];
  auto fetch_norm = [&](const uint16_t* weight, const uint16_t* bias) MODA_INLINE {
#pragma unroll
    for (int j = 0; j < NL; j++) {
      wv[j] = *reinterpret_cast<const i32x4*>(weight + (lsub + TPR * j) * 8);
      bv[j] = *reinterpret_cast<const i32x4*>(bias + (lsub + TPR * j) * 8);
    }
  };
  auto layer_norm = [&](bool normalise, float eps, uint16_t* out) MODA_INLINE {
    auto load8 = [](const i32x4& v, float (&f)[8]) {
#pragma unroll
      for (int i = 0; i < 4; i++) unpack2<T>(v[i], f[2 * i], f[2 * i + 1]);
    };
    lds_barrier();
    float f[NL][8], s[NL];
    i32x4 raw[NL];
#pragma unroll
    for (int j = 0; j < NL; j++) {
      raw[j] = *reinterpret_cast<MODA_LDS const i32x4*>(X + Rows<C>::off(lrow, lsub + TPR * j));
      load8(raw[j], f[j]);
      s[j] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) s[j] += f[j][i];
    }
    const bool store = out && r0 + lrow < rows_end;
    if (!POST && store) {
#pragma unroll
      for (int j = 0; j < NL; j++) *reinterpret_cast<i32x4*>(out + (int64_t)(r0 + lrow) * C + (lsub + TPR * j) * 8) = raw[j];
    }
    if (normalise) {
      const float mean = row_sum<TPR>(s) / C;
#pragma unroll
      for (int j = 0; j < NL; j++) {
        s[j] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float d = f[j][i] - mean;
          s[j] = __builtin_fmaf(d, d, s[j]);
        }
      }
      const float rstd = rsqrtf(row_sum<TPR>(s) / C + eps);
#pragma unroll
      for (int j = 0; j < NL; j++) {
        float w[8], b[8];
        load8(wv[j], w);
        load8(bv[j], b);
        i32x4 o;
#pragma unroll
        for (int i = 0; i < 4; i++)
          o[i] = pack2<T>((f[j][2 * i] - mean) * rstd * w[2 * i] + b[2 * i], (f[j][2 * i + 1] - mean) * rstd * w[2 * i + 1] + b[2 * i + 1]);
        *reinterpret_cast<MODA_LDS i32x4*>(X + Rows<C>::off(lrow, lsub + TPR * j)) = o;
        if (POST && store) *reinterpret_cast<i32x4*>(out + (int64_t)(r0 + lrow) * C + (lsub + TPR * j) * 8) = o;
      }
    }
    lds_barrier();
  };

  auto read_keep = [&]() MODA_INLINE {
#pragma unroll
    for (int mb = 0; mb < MB2; mb++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++) keep[mb][nb] = *reinterpret_cast<MODA_LDS const i32x2*>(own_piece(mb, nb));
  };
  zero(acc);
  proj.template run<C>(H, xbase, C / 32, acc);
  read_keep();  // (the pieces that add_keep overwrites are the ones this lane reads)
  // this wave's features of the hidden chunk that starts at c0: f1 = c0 + wave * 16 * MB1, none in a short last chunk
  Product<T, MB1, NB> fc1;
  fc1.voff = lane * 16;
  i32x2 bias1[MB1];
  auto has_features = [&](int c0) { return c0 + wave * 16 * MB1 < a.hidden; };
  auto start_fc1 = [&](int c0) MODA_INLINE {
    // BESIDE: the waves that a short last chunk has no features for take others' and keep the result to themselves
    if (!BESIDE && !has_features(c0)) return;
    const int f1 = !BESIDE || has_features(c0) ? c0 + wave * 16 * MB1 : c0;
#pragma unroll
    for (int mb = 0; mb < MB1; mb++) fc1.base[mb] = a.fc1_w + (size_t)(f1 + 16 * mb) * C;
    fc1.start();
    pieces(a.fc1_b, f1, bias1);
  };
  start_fc1(0);
  fetch_norm(a.mid_w, a.mid_b);
  add_keep();
  layer_norm(true, a.mid_eps, nullptr);
  if (POST) read_keep();

  // MLP, HC hidden features at a time; two stages of hidden activations, so that one barrier a chunk is enough
  zero(acc);
  Product<T, MB2, NB> fc2;
  fc2.voff = lane * 16;
  lds_ptr Hs = H;
  // piece (mb, nb) of a chunk's first product: bias, activation, into the stage `to`
  auto activate = [&](const f32x4& sum, const float (&b)[4], int mb, int nb, lds_ptr to) MODA_INLINE {
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = sum[i] + b[i];
    i32x2 w = pack4(x);  // the linear layer's own result is a 16-bit value, as it is when the layers run one by one
    w[0] = activated<T>(w[0], table);
    w[1] = activated<T>(w[1], table);
    *reinterpret_cast<MODA_LDS i32x2*>(to + Rows<HC>::off(sigma, wave * 2 * MB1 + 2 * mb + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * HC) = w;
  };
  auto fc2_at = [&](int c0) MODA_INLINE {
#pragma unroll
    for (int mb = 0; mb < MB2; mb++) fc2.base[mb] = a.fc2_w + (size_t)(f2 + 16 * mb) * a.hidden + c0 * 16;
  };
  if constexpr (BESIDE) {
    static_assert(Product<T, MB1, NB>::PF == Product<T, MB2, NB>::PF && C / 32 >= Product<T, MB1, NB>::PF, "as many steps on their way in both");
    constexpr int PF = Product<T, MB1, NB>::PF, N1 = C / 32, N2 = HC / 32;
    static_assert(N2 >= MB1 * NB, "a step for every piece");
    f32x4 hid[MB1][NB];
    zero(hid);
    fc2_at(0);
    fc1.template run_beside<C, N1>(X, xbase, hid, [&](int j) MODA_INLINE {
      if (j >= N1 - PF) fc2.load(j - (N1 - PF));
    });
    if (has_features(0))
#pragma unroll
      for (int mb = 0; mb < MB1; mb++) {
        float b[4];
        unpack4(bias1[mb], b);
#pragma unroll
        for (int nb = 0; nb < NB; nb++) activate(hid[mb][nb], b, mb, nb, Hs);
      }
    for (int c0 = 0; c0 + HC < a.hidden; c0 += HC) {
      lds_ptr other = Hs == H ? H + BM * HC : H;
      start_fc1(c0 + HC);
      lds_barrier();
      zero(hid);
      fc1.template run_beside<C, N1>(X, xbase, hid, [](int) {});
      const bool mine = has_features(c0 + HC);
      fc2.template run_beside<HC, N2>(Hs, hbase, acc, [&](int j) MODA_INLINE {
        if (j >= MB1 * NB || !mine) return;
        float b[4];
        unpack4(bias1[j / NB], b);
        activate(hid[j / NB][j % NB], b, j / NB, j % NB, other);
      });
      fc2_at(c0 + HC);
      fc2.start();
      Hs = other;
    }
    lds_barrier();
    fc2.template run<HC>(Hs, hbase, ((a.hidden - 1) % HC + 1) / 32, acc);
  } else {
    for (int c0 = 0; c0 < a.hidden; c0 += HC) {
      if (has_features(c0)) {
        f32x4 hid[MB1][NB];
        zero(hid);
        fc1.template run<C>(X, xbase, C / 32, hid);
#pragma unroll
        for (int mb = 0; mb < MB1; mb++) {
          float b[4];
          unpack4(bias1[mb], b);
#pragma unroll
          for (int nb = 0; nb < NB; nb++) activate(hid[mb][nb], b, mb, nb, Hs);
        }
      }
#pragma unroll
      for (int mb = 0; mb < MB2; mb++) fc2.base[mb] = a.fc2_w + (size_t)(f2 + 16 * mb) * a.hidden + c0 * 16;  // (fc2_at: 4 registers more)
      fc2.start();
      lds_barrier();
      const int left = a.hidden - c0;
      fc2.template run<HC>(Hs, hbase, (left < HC ? left : HC) / 32, acc);
      if (c0 + HC < a.hidden) start_fc1(c0 + HC);
      Hs = Hs == H ? H + BM * HC : H;
    }
  }
  pieces(a.fc2_b, f2, bias2);
  const bool end_norm = POST || a.n_parts > 0;
  if (end_norm) fetch_norm(a.end_w, a.end_b);
  add_keep();
  layer_norm(end_norm, a.end_eps, a.x);
  if (a.n_parts == 0) return;

  // Projections of the next block: 8 MBQ blocks of 16 features a turn, MBQ a wave, so many that one turn is enough where
  // four are.  Results leave through LDS, by rows.
  const int end0 = a.part[0].block_end, end1 = a.n_parts > 1 ? a.part[1].block_end : end0, blocks = a.part[a.n_parts - 1].block_end;
  auto projections = [&](auto side_by_side) MODA_INLINE {
    constexpr int MBQ = decltype(side_by_side)::value, W = 128 * MBQ;
#pragma unroll 1
    for (int first = 0; first < blocks; first += 8 * MBQ) {
      Product<T, MBQ, NB> next;
      next.voff = lane * 16;
      i32x2 bias[MBQ];
#pragma unroll
      for (int mb = 0; mb < MBQ; mb++) {
        const int want = first + wave * MBQ + mb, blk = want < blocks ? want : blocks - 1;  // past the last block: that one again, not stored
        const int pi = blk < end0 ? 0 : blk < end1 ? 1 : 2, f = 16 * (blk - (pi == 0 ? 0 : pi == 1 ? end0 : end1));
        next.base[mb] = (pi == 0 ? a.part[0].w : pi == 1 ? a.part[1].w : a.part[2].w) + (size_t)f * C;
        const uint16_t* bp = pi == 0 ? a.part[0].bias : pi == 1 ? a.part[1].bias : a.part[2].bias;
        bias[mb] = bp ? *reinterpret_cast<const i32x2*>(bp + f + 4 * q4) : none;
      }
      next.start();
      if (first > 0) lds_barrier();  // the results of the turn before are read
      f32x4 out[MBQ][NB];
      zero(out);
      next.template run<C>(X, xbase, C / 32, out);
#pragma unroll
      for (int mb = 0; mb < MBQ; mb++) {
        float b[4];
        unpack4(bias[mb], b);
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = out[mb][nb][i] + b[i];
          *reinterpret_cast<MODA_LDS i32x2*>(H + Rows<W>::off(sigma, 2 * (wave * MBQ + mb) + (q4 >> 1)) + 4 * (q4 & 1) + 16 * nb * W) = pack4(x);
        }
      }
      lds_barrier();
      const int chunks = 2 * (blocks - first < 8 * MBQ ? blocks - first : 8 * MBQ);  // of 8 features a row
      if (r0 + lrow < rows_end)
#pragma unroll 2
        for (int ch = lsub; ch < chunks; ch += TPR) {
          const int blk = first + (ch >> 1), f = 8 * (2 * first + ch);
          uint16_t* y = blk < end0 ? a.part[0].y + f : blk < end1 ? a.part[1].y + (f - 16 * end0) : a.part[2].y + (f - 16 * end1);
          const int64_t ldy = blk < end0 ? a.part[0].ldy : blk < end1 ? a.part[1].ldy : a.part[2].ldy;
          *reinterpret_cast<i32x4*>(y + (r0 + lrow) * ldy) = *reinterpret_cast<MODA_LDS const i32x4*>(H + Rows<W>::off(lrow, ch));
        }
    }
  };
  if (blocks <= 16)
    projections(std::integral_constant<int, 2>{});
  else if (blocks <= 24)
    projections(std::integral_constant<int, 3>{});
  else
    projections(std::integral_constant<int, 4>{});
}

inline TailArgs tail_args(const moda_hip_block_tail_args* t) {
  TailArgs a = {};
  auto in = [](const void* p) { return (const uint16_t*)p; };
  a.h = in(t->attention);
  a.res = in(t->residual);
  a.x = (uint16_t*)t->x;
  a.rows = (int)t->rows;
  a.hidden = (int)t->hidden;
  a.n_parts = t->n_parts;
  a.proj_w = in(t->proj_w);
  a.proj_b = in(t->proj_b);
  a.fc1_w = in(t->fc1_w);
  a.fc1_b = in(t->fc1_b);
  a.fc2_w = in(t->fc2_w);
  a.fc2_b = in(t->fc2_b);
  a.mid_w = in(t->mid_norm_w);
  a.mid_b = in(t->mid_norm_b);
  a.end_w = in(t->end_norm_w);
  a.end_b = in(t->end_norm_b);
  a.mid_eps = t->mid_norm_eps;
  a.end_eps = t->end_norm_eps;
  a.gelu_table = (const float*)t->gelu_table;
  int end = 0;
  for (int i = 0; i < t->n_parts; i++) {
    const moda_hip_linear_part& p = t->parts[i];
    end += (int)p.n / 16;
    a.part[i] = TailPart{in(p.w), in(p.bias), (uint16_t*)p.y, p.ldy, end};
  }
  return a;
}

}  // namespace moda
