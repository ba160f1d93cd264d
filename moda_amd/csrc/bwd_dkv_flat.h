// Backward, key side, sequence keys on the 64-wide tiles where the key head is the query head, fixed-length and packed: the
// same products as dkv_kernel (moda_v14.py:874-1248, fla/ops/attn/parallel.py:299-440) without the split into two roles.
//
// A workgroup of FOUR waves owns 128 key columns of one (batch, kv head), a wave 32 of them with K AND V in
// registers and BOTH accumulators, dK^T and dV^T; the query rows come by in tiles of 32 (one summation step of the
// 16x16x32 instruction):
//   S = Q K^T, dP - delta = dO V^T (accumulators preset with -delta), P = exp2(S c - lse), dS = P (dP - delta),
//   dV^T += dO^T P, dK^T += Q^T dS.
// P stays in fp32 until dS is formed (one rounding on the dK path) and nothing travels between waves.  With 26 KB of
// LDS and no mailbox, three workgroups share a compute unit where dkv_kernel fits one: twelve waves per compute unit
// instead of eight cover each other's softmax, start and end.  On the 128-wide tiles this structure spills.
//
// SPLIT: the query rows of long column tiles are cut into segments of about equal length (geometry.h: dkv_split_plan),
// which leave fp32 partial sums for dkv_reduce_kernel: without them the launch ends with the heaviest tile.
//
// RW (row waves): the four waves share the SAME 32 columns and take 32 rows each of every 128-row query tile; their
// accumulators meet in LDS, in wave order, before the rows are written.  For short launches with too few 128-column
// tiles to fill the machine (geometry.h: dkv_flat_row_waves): four times the workgroups, a quarter of the trips.
#pragma once
#include <type_traits>

#include "geometry.h"
#include "kargs.h"
#include "tile.h"
#include "tile16.h"

namespace moda {

// VARLEN: packed variable-length batch (a workgroup enters its sequence; column tiles past its end leave at once)
// As a kernel of its own or, MODA_SIDE_BY_SIDE, as a function (see dq_kernel); `block` is the workgroup's place among these
// OWN_DELTA: the row sums of o * do are formed here, tile by tile (a launch that runs beside the dQ kernel's workgroups
// cannot read theirs); the same additions in the same order as there
template <typename T, int HD, bool VARLEN, bool SPLIT, int RW = 1, bool OWN_DELTA = false>
#ifdef MODA_SIDE_BY_SIDE
__device__ __forceinline__ void dkv_flat_body(const KArgs& a_in, int block) {
#else
__global__ __launch_bounds__(256, RW == 1 ? 3 : 2) void dkv_flat_kernel(const KArgs a_in) {
  const int block = blockIdx.x;
#endif
  static_assert(RW == 1 || (RW == 4 && !VARLEN && !SPLIT), "four row waves: fixed length, no segments");
  static_assert(!OWN_DELTA || (RW == 4 && HD == 64), "row sums of launches with row waves, eight chunks a row");
  constexpr int NB = 2, WM = 32, BM = WM * RW, MBLK = WM / 16, BN = 4 / RW * 16 * NB, KS = HD / 32, MB = HD / 16;
  constexpr int NST = RW == 1 ? 3 : 2, DIST = NST - 1;  // ring stages, tiles in flight
  constexpr int SP = RW == 1 ? 64 : BM;  // floats per statistic and stage (wave-wide loads)
  extern __shared__ __align__(16) unsigned char smem_raw[];
  lds_ptr ring = (lds_ptr)smem_raw;                                      // [NST]: Q tile, dO tile
  MODA_LDS float* stat = (MODA_LDS float*)(ring + NST * 2 * BM * HD);    // [NST][2][SP]: lse, minus delta
  MODA_LDS float* own_stat = stat + NST * 2 * SP + (threadIdx.x >> 6) * WM;  // OWN_DELTA: [4][WM], a wave's own rows

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ColPlace place = col_place<VARLEN>(a_in, (int)block, BN, SPLIT ? a_in.dkv_split : 1);
  if (VARLEN && !place.active) return;
  const int ct = place.ct, hkv = place.hkv;
  int b = place.b;
  SeqArgs<VARLEN> seq(a_in, b, place.t0, place.T);
  const KArgs& a = seq.a;
  const ColTilePlan plan = col_tile_plan(a_in, a, ct, BN, BM, VARLEN, SPLIT ? a.dkv_split : 1);
  if ((VARLEN || SPLIT) && !plan.active) return;  // a tile beyond its sequence, or a segment beyond its tile
  const int cw = RW == 1 ? wave : 0, rw = RW == 1 ? 0 : wave;  // the wave's column block, its rows of a query tile
  int c[NB];
  bool valid[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    c[nb] = plan.c_first + cw * (16 * NB) + 16 * nb + n;
    valid[nb] = c[nb] < a.T;
  }
  i32x4 Kr[NB][KS], Vr[NB][KS];
  {
    const uint16_t* kp = a.k + b * a.sk.b + hkv * a.sk.h + 8 * q4;
    const uint16_t* vp = a.v + b * a.sv.b + hkv * a.sv.h + 8 * q4;
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        i32x4 z = {0, 0, 0, 0};
        Kr[nb][ks] = (valid[nb] && 32 * ks + 8 * q4 < a.D) ? *reinterpret_cast<const i32x4*>(kp + (int64_t)c[nb] * a.sk.t + 32 * ks) : z;
        Vr[nb][ks] = (valid[nb] && 32 * ks + 8 * q4 < a.Dv) ? *reinterpret_cast<const i32x4*>(vp + (int64_t)c[nb] * a.sv.t + 32 * ks) : z;
      }
  }
  // No wait here: K and V travel together with the first query tiles.  The compiler waits for all loads it knows
  // of before the first product, which (loads returning in order) also covers nothing it does not know of.

  int qlo[NB], qhi[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    qlo[nb] = qhi[nb] = 0;
    if (valid[nb]) q_interval(a, false, c[nb], qlo[nb], qhi[nb]);
  }
  const int qt0 = plan.qt0, nqt = plan.nqt;

  typedef AsyncTileLoader<HD, BM, 256> Loader;
  constexpr int LPT = 2 * Loader::N + 1;  // vector-memory loads one wave issues per tile: Q, dO and one statistic
  Loader ld;
  ld.init(tid);
  const uint16_t* qb = a.q + b * a.sq.b + hkv * a.sq.h;
  const uint16_t* dob = a.d_o + b * a.sdo.b + hkv * a.sdo.h;
  // even waves fetch lse ([B, Tq, Hq]: one dword every Hq), odd waves minus delta ([B, Hq, Tq]: contiguous); the two
  // waves of a kind write the same values to the same place, which keeps every wave's load count per tile equal
  const bool st_lse = OWN_DELTA || (wave & 1) == 0;
  const char* stb = st_lse ? (const char*)(a.lse + (int64_t)b * a.Tq * a.Hq + hkv) : (const char*)(a.delta + ((int64_t)b * a.Hq + hkv) * (VARLEN ? a.delta_pitch : a.Tq));
  const uint32_t st_row = st_lse ? (uint32_t)a.Hq * 4u : 4u;
  const int st_first = SP == 64 ? 0 : (wave >> 1) * 64;  // first row this wave fetches of a tile's statistics
  const int voff_stat = (st_first + lane) * (int)st_row;
  int ld_st = 0;
  auto issue = [&](int it) {  // trip `it` consumes query tile nqt - 1 - it
    const int f_q0 = (qt0 + nqt - 1 - it) * BM;
    lds_ptr Qt = ring + ld_st * 2 * BM * HD;
    ld.load(Qt, qb, a.sq.t, f_q0, a.Tq, a.D);
    ld.load(Qt + BM * HD, dob, a.sdo.t, f_q0, a.Tq, a.Dv);
    const int rows = imax(imin(a.Tq - f_q0, BM), 0);
    const i32x4 rs = rsrc_words(stb + (int64_t)f_q0 * st_row, rows > 0 ? (uint32_t)(rows - 1) * st_row + 4u : 0u);
    lds_dma<4>(rs, (uint32_t)(uintptr_t)(stat + ld_st * 2 * SP + (st_lse ? 0 : SP) + st_first), voff_stat, 0);
    ld_st = (ld_st + 1 == NST) ? 0 : ld_st + 1;
  };
  auto wait_tile = [&](int next) {
    if (DIST == 2 && next + 1 < nqt)
      Loader::template wait_but<LPT>();
    else
      Loader::wait_all();
  };

  f32x4 dk[MB][NB], dv[MB][NB];
#pragma unroll
  for (int d = 0; d < MB; d++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) dk[d][nb] = dv[d][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale * kLog2e;
  Operand16<HD> oa;
  oa.init(lane);

  // OWN_DELTA: two lanes a row of the wave's 32; pieces of o that go with lane groups q = 2 half and 2 half + 1 of the dQ
  // kernel.  They are fetched a tile ahead.
  const int own_row = lane >> 1, own_half = lane & 1;
  auto own_chunk = [&](int c) { return 2 * own_half + (c >> 1) + 4 * (c & 1); };
  i32x4 o_piece[4];
  auto fetch_o = [&](int it) {
    const int r = imin((qt0 + nqt - 1 - it) * BM + rw * WM + own_row, a.Tq - 1);
    const uint16_t* row = a.o + b * a.so.b + hkv * a.so.h + (int64_t)r * a.so.t;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const bool in = own_chunk(c) * 8 < a.Dv;
      const i32x4 v = *reinterpret_cast<const i32x4*>(row + (in ? own_chunk(c) * 8 : 0)), z = {0, 0, 0, 0};
      o_piece[c] = in ? v : z;
    }
  };
  if (OWN_DELTA && nqt > 0) fetch_o(0);
#pragma unroll
  for (int j = 0; j < DIST; j++)
    if (j < nqt) issue(j);
  wait_tile(0);
  __syncthreads();

  auto tile = [&](auto masked, int st, int it) {
    const int q0 = (qt0 + nqt - 1 - it) * BM;
    constexpr bool MASKED = decltype(masked)::value;
    lds_cptr Qs = ring + st * 2 * BM * HD + rw * (WM * HD);
    lds_cptr dOs = Qs + BM * HD;
    MODA_LDS const float* lse_s = stat + st * 2 * SP + rw * WM;
    MODA_LDS const float* del_s = OWN_DELTA ? (MODA_LDS const float*)own_stat : lse_s + SP;
    if (OWN_DELTA) {
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const i32x4 d = *reinterpret_cast<MODA_LDS const i32x4*>(dOs + Tile<HD>::off(own_row, own_chunk(c)));
#pragma unroll
        for (int w = 0; w < 4; w++) {
          float x0, x1, y0, y1;
          unpack2<T>(o_piece[c][w], x0, x1);
          unpack2<T>(d[w], y0, y1);
          sum[c >> 1] = __builtin_fmaf(x0, y0, sum[c >> 1]);
          sum[c >> 1] = __builtin_fmaf(x1, y1, sum[c >> 1]);
        }
      }
      float row_sum = sum[0] + sum[1];
      row_sum += __shfl_xor(row_sum, 1, 64);
      // a row past the end has zeros everywhere, though the last row's o was read for it
      if (own_half == 0) own_stat[own_row] = q0 + rw * WM + own_row < a.Tq ? -row_sum : 0.f;
      if (it + 1 < nqt) fetch_o(it + 1);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // the wave reads what its lanes wrote
      asm volatile("" ::: "memory");
    }
    f32x4 s[MBLK][NB], dp[MBLK][NB];
#pragma unroll
    for (int m = 0; m < MBLK; m++) {
      const f32x4 dl = *reinterpret_cast<MODA_LDS const f32x4*>(del_s + 16 * m + slot_base(q4));
#pragma unroll
      for (int nb = 0; nb < NB; nb++) dp[m][nb] = dl;
    }
    {  // S and dP in one pipeline, two operand reads ahead of the matrix pipe
      constexpr int N = 2 * MBLK * KS, DEPTH = 2;
      i32x4 ops[N];
      auto rd = [&](int j) { return oa.row_operand((j & 1) ? dOs : Qs, 16 * ((j >> 1) % MBLK), (j >> 1) / MBLK); };
#pragma unroll
      for (int j = 0; j < DEPTH; j++) ops[j] = rd(j);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < N; j++) {
        if (j + DEPTH < N) ops[j + DEPTH] = rd(j + DEPTH);
        const int m = (j >> 1) % MBLK, ks = (j >> 1) / MBLK;
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
          if (j & 1)
            dp[m][nb] = mfma16<T>(ops[j], Vr[nb][ks], dp[m][nb]);
          else
            s[m][nb] = mfma16<T>(ops[j], Kr[nb][ks], ks == 0 ? z : s[m][nb]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    TrPipe16<T, HD, 1, NB, 3> pv;
    pv.prefetch(oa, dOs);
#pragma unroll
    for (int m = 0; m < MBLK; m++) {
      const f32x4 lv = *reinterpret_cast<MODA_LDS const f32x4*>(lse_s + 16 * m + slot_base(q4));
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float p = fast_exp2(__builtin_fmaf(s[m][nb][j], sc, -lv[j]));
          if (MASKED) {
            const int qr = q0 + rw * WM + 16 * m + slot_base(q4) + j;
            p = (qr >= qlo[nb] && qr < qhi[nb]) ? p : 0.f;
          }
          s[m][nb][j] = p;
          dp[m][nb][j] *= p;
        }
    }
    i32x4 P[1][NB], DS[1][NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      P[0][nb] = pack_slots<T>(s[0][nb], s[1][nb]);
      DS[0][nb] = pack_slots<T>(dp[0][nb], dp[1][nb]);
    }
    pv.run(oa, dOs, P, dv);
    TrPipe16<T, HD, 1, NB, 3> pk;
    pk.prefetch(oa, Qs);
    pk.run(oa, Qs, DS, dk);
  };

  // query tiles whose rows all see all columns of the workgroup need no masking: for causal keys those at or past the last
  // column's first visible row (padding rows past Tq carry zero Q, dO, lse, delta and contribute nothing)
  const int first_free_qt = a.causal ? ((imin(a.T, plan.c_first + BN) - 1) * a.Gf + BM - 1) / BM - qt0 : 0;
  int it = 0, c_st = 0;
  for (; it < nqt && nqt - 1 - it >= first_free_qt; it++) {
    if (it + DIST < nqt) issue(it + DIST);
    tile(std::false_type{}, c_st, it);
    c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    wait_tile(it + 1);
    __syncthreads();
  }
  for (; it < nqt; it++) {
    if (it + DIST < nqt) issue(it + DIST);
    tile(std::true_type{}, c_st, it);
    c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    wait_tile(it + 1);
    __syncthreads();
  }

  auto own_slot_row = [&](bool is_v, int col) -> const uint16_t* {  // this lane's part of slot Lv of the column's token
    const int64_t row = (int64_t)col * a.L + a.Lv;
    return (is_v ? a.dvd + b * a.sdvd.b + hkv * a.sdvd.h + row * a.sdvd.t : a.dkd + b * a.sdkd.b + hkv * a.sdkd.h + row * a.sdkd.t) + 4 * q4;
  };
  auto add_own = [&](f32x4& x, const i32x2& w) {
    float f[4];
    unpack2<T>(w[0], f[0], f[1]);
    unpack2<T>(w[1], f[2], f[3]);
    x += f32x4{f[0], f[1], f[2], f[3]};
  };
  if constexpr (RW > 1) {
    // [which][d][nb] blocks of all waves through the ring (which every wave has done reading): wave w adds up and writes
    // a quarter of them
    static_assert(NST * 2 * BM * HD * 2 >= 4 * 2 * MB * NB * 1024 && 2 * MB % RW == 0, "the exchange fits the ring");
    MODA_LDS f32x4* ex = (MODA_LDS f32x4*)ring;
#pragma unroll
    for (int d = 0; d < MB; d++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        ex[((rw * 2 * MB + d) * NB + nb) * 64 + lane] = dk[d][nb];
        ex[((rw * 2 * MB + MB + d) * NB + nb) * 64 + lane] = dv[d][nb];
      }
    const bool is_v = rw >= RW / 2;
    i32x2 own[NB][2 * MB / RW];  // the layer's own slot: on its way while the accumulators are exchanged
    if (a.own_slot) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const uint16_t* slot = own_slot_row(is_v, c[nb]);
#pragma unroll
        for (int i = 0; i < 2 * MB / RW; i++) {
          const int d = (rw * (2 * MB / RW) + i) % MB;
          own[nb][i] = valid[nb] && 16 * d + 4 * q4 < (is_v ? a.Dv : a.D) ? *reinterpret_cast<const i32x2*>(slot + 16 * d) : i32x2{0, 0};
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      uint16_t* outp = is_v ? a.dv + b * a.sdv.b + hkv * a.sdv.h + (int64_t)c[nb] * a.sdv.t
                            : a.dk + b * a.sdk.b + hkv * a.sdk.h + (int64_t)c[nb] * a.sdk.t;
#pragma unroll
      for (int i = 0; i < 2 * MB / RW; i++) {
        const int blk = rw * (2 * MB / RW) + i, d = blk % MB;
        f32x4 sum = ex[(blk * NB + nb) * 64 + lane];
#pragma unroll
        for (int w = 1; w < RW; w++) sum += ex[((w * 2 * MB + blk) * NB + nb) * 64 + lane];
        sum *= is_v ? 1.f : a.scale;
        if (a.own_slot) add_own(sum, own[nb][i]);
        i32x2 w;
        w[0] = pack2<T>(sum[0], sum[1]);
        w[1] = pack2<T>(sum[2], sum[3]);
        if (valid[nb] && 16 * d + 4 * q4 < (is_v ? a.Dv : a.D)) *reinterpret_cast<i32x2*>(outp + 16 * d + 4 * q4) = w;
      }
    }
    return;
  }
  if (SPLIT && plan.nsegs > 1) {  // a row segment: fp32 partial sums, added up by dkv_reduce_kernel
    const int64_t pitch = part_rows(a), plane = (int64_t)(VARLEN ? 1 : a.B) * a.Hkv * pitch * HD;
    const int first = VARLEN ? place.t0 : 0;
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
      if (valid[nb]) {
        float* kp = a.dkv_part + plan.seg * plane + (((int64_t)b * a.Hkv + hkv) * pitch + first + c[nb]) * HD + 4 * q4;
        float* vp = kp + a.dkv_split * plane;
#pragma unroll
        for (int d = 0; d < MB; d++) {
          *reinterpret_cast<f32x4*>(kp + 16 * d) = dk[d][nb] * a.scale;
          *reinterpret_cast<f32x4*>(vp + 16 * d) = dv[d][nb];
        }
      }
    return;
  }
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
    if (valid[nb]) {
      uint16_t* dkp = a.dk + b * a.sdk.b + hkv * a.sdk.h + (int64_t)c[nb] * a.sdk.t + 4 * q4;
      uint16_t* dvp = a.dv + b * a.sdv.b + hkv * a.sdv.h + (int64_t)c[nb] * a.sdv.t + 4 * q4;
#pragma unroll
      for (int d = 0; d < MB; d++) {
        if (SPLIT) dk[d][nb] *= a.scale;
        if (SPLIT && !VARLEN && a.own_slot) {  // (not in the instantiation of the long launches: 0.7 % of their time)
          if (16 * d + 4 * q4 < a.D) add_own(dk[d][nb], *reinterpret_cast<const i32x2*>(own_slot_row(false, c[nb]) + 16 * d));
          if (16 * d + 4 * q4 < a.Dv) add_own(dv[d][nb], *reinterpret_cast<const i32x2*>(own_slot_row(true, c[nb]) + 16 * d));
        }
        i32x2 w;
        const float mul = SPLIT ? 1.f : a.scale;
        w[0] = pack2<T>(dk[d][nb][0] * mul, dk[d][nb][1] * mul);
        w[1] = pack2<T>(dk[d][nb][2] * mul, dk[d][nb][3] * mul);
        if (16 * d + 4 * q4 < a.D) *reinterpret_cast<i32x2*>(dkp + 16 * d) = w;
        w[0] = pack2<T>(dv[d][nb][0], dv[d][nb][1]);
        w[1] = pack2<T>(dv[d][nb][2], dv[d][nb][3]);
        if (16 * d + 4 * q4 < a.Dv) *reinterpret_cast<i32x2*>(dvp + 16 * d) = w;
      }
    }
}

// LDS of a workgroup
template <int HD, int RW, bool OWN_DELTA>
constexpr size_t dkv_flat_lds() {
  return (RW == 1 ? (size_t)3 * (2 * 32 * HD * sizeof(uint16_t) + 2 * 64 * sizeof(float))
                  : (size_t)2 * (2 * 32 * RW * HD * sizeof(uint16_t) + 2 * 32 * RW * sizeof(float))) +
         (OWN_DELTA ? 4 * 32 * sizeof(float) : 0);
}

}  // namespace moda
