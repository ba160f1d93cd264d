// Backward, query side: the body of the dQ kernel (bwd_dq_kernel.hip has what it computes and how it is laid out).
#pragma once
#include <type_traits>

#include "geometry.h"
#include "kargs.h"
#include "tile.h"
#include "tile16.h"
#include "tuning.h"

namespace moda {

// ADDR bit 0: a (batch, head) slice is wider than 2 GiB (descriptors anchored per tile instead of 32-bit
// offsets inside the slice); bit 1: packed variable-length batch; bit 2: no depth stream; bit 3: partially filled
// depth stream (only Lv of a token's L slots hold data: depth tiles are loaded through the slot mapping)
// The body is a kernel of its own, or (MODA_SIDE_BY_SIDE, bwd_short_kernel.hip) a function whose workgroups share a launch with
// others; `block` is the workgroup's place among the dQ workgroups.  A kernel that calls the function is not the same code: its
// inlined body is optimised once by itself, without the argument block's values, and took 3.70 against 3.60 ms at 16 K tokens,
// 64 query heads, 64 slots (dkv_flat_kernel 5.17 against 4.30).
template <typename T, int HD, typename Shape, int ADDR>
#ifdef MODA_SIDE_BY_SIDE
__device__ __forceinline__ void dq_body(const KArgs& a_in, int block) {
#else
__global__ __launch_bounds__(64 * Shape::W, 2) void dq_kernel(const KArgs a_in) {
  const int block = blockIdx.x;
#endif
  constexpr int NB = Shape::NB, WR = 16 * NB, BM = WR * Shape::W, BN = 64, KS = HD / 32, MB = HD / 16, NT = 64 * Shape::W, NST = Shape::NST, DIST = Shape::DIST;
  static_assert(NST >= DIST + 1 && DIST >= 1 && DIST <= 2, "ring must hold the tile in use plus the tiles in flight");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  lds_ptr smem = (lds_ptr)smem_raw;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, q4 = lane >> 4;
  constexpr bool WIDE = (ADDR & 1) != 0, VARLEN = (ADDR & 2) != 0;
  // bit 2: launched without a depth stream (the plain and sequence-only calls): the depth code is compiled out,
  // so that it cannot disturb the register allocation of their main loop
  constexpr bool NODEPTH = (ADDR & 4) != 0, PARTIAL = (ADDR & 8) != 0;
  static_assert(!(NODEPTH && PARTIAL), "a partially filled depth stream is a depth stream");
  const RowPlace place = row_place<VARLEN>(a_in, (int)block, BM);
  if (VARLEN && !place.active) return;
  int b = place.b;
  const int hq = place.hq, hkv = hq / a_in.hdiv, qt = place.qt;
  SeqArgs<VARLEN> seq(a_in, b, place.t0, place.T);
  const KArgs& a = seq.a;
  const int Ld = NODEPTH ? 0 : a.L;  // depth slots per token

  // Loads of the row operands and, on the 64-wide tiles with depth, of o, which has the row sums wait for it: the first tiles of
  // the ring are sent for in between, so that all of it travels together.  Those take their masked tiles by halves, too.  Without
  // depth neither pays: training steps of 8 x 1200 tokens, four heads of four, causal, 191 us with both, 188 with whole tiles and
  // 186 with neither; 16 x 577, six of two, 102, 100 and 100.
  constexpr bool HALVES = HD <= 64 && !NODEPTH, SUMS_LATE = HALVES;
  i32x4 Qr[NB][KS], dOr[NB][KS], Or[NB][KS];
  float lse[NB], delta[NB];
  int shi[NB], dlo[NB], dhi[NB];
  auto load_o = [&](int nb) {
    const int r = qt * BM + wave * WR + 16 * nb + n;
    const uint16_t* orow = a.o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t + 8 * q4;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      i32x4 z = {0, 0, 0, 0};
      Or[nb][ks] = (r < a.Tq && 32 * ks + 8 * q4 < a.Dv) ? *reinterpret_cast<const i32x4*>(orow + 32 * ks) : z;
    }
  };
  auto row_sum = [&](int nb) {
    const int r = qt * BM + wave * WR + 16 * nb + n;
    const bool valid = r < a.Tq;
    float* drow = a.delta + ((int64_t)b * a.Hq + hq) * (VARLEN ? a.delta_pitch : a.Tq) + r;
    delta[nb] = 0.f;
    if (a.own_delta) {
      // minus rowsum(o * do) (moda_v14.py:525-539) from the dO pieces this lane holds anyway and the same pieces of
      // o; the four lanes of a row add their shares and the first one leaves the sum for the kernels that follow
      if (!SUMS_LATE) load_o(nb);
      float acc = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
          float x0, x1, y0, y1;
          unpack2<T>(Or[nb][ks][w], x0, x1);
          unpack2<T>(dOr[nb][ks][w], y0, y1);
          acc = __builtin_fmaf(x0, y0, acc);
          acc = __builtin_fmaf(x1, y1, acc);
        }
      acc = quad_sum(acc);
      delta[nb] = valid ? -acc : 0.f;
      if (valid && q4 == 0) *drow = -acc;
    } else if (valid) {
      delta[nb] = *drow;
    }
  };
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const int r = qt * BM + wave * WR + 16 * nb + n;
    const bool valid = r < a.Tq;
    const uint16_t* qp = a.q + b * a.sq.b + hq * a.sq.h + (int64_t)r * a.sq.t + 8 * q4;
    const uint16_t* dop = a.d_o + b * a.sdo.b + hq * a.sdo.h + (int64_t)r * a.sdo.t + 8 * q4;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      i32x4 z = {0, 0, 0, 0};
      Qr[nb][ks] = (valid && 32 * ks + 8 * q4 < a.D) ? *reinterpret_cast<const i32x4*>(qp + 32 * ks) : z;
      dOr[nb][ks] = (valid && 32 * ks + 8 * q4 < a.Dv) ? *reinterpret_cast<const i32x4*>(dop + 32 * ks) : z;
    }
    lse[nb] = 0.f;
    if (valid) lse[nb] = a.lse[((int64_t)b * a.Tq + r) * a.Hq + hq];
    if (!SUMS_LATE)
      row_sum(nb);
    else if (a.own_delta)
      load_o(nb);
    const RowVis vis = row_visibility(a, r, Ld);
    shi[nb] = vis.shi;
    dlo[nb] = vis.dlo;
    dhi[nb] = vis.dhi;
  }
  // Depth columns a wave alone can see are not streamed through the workgroup's ring: each wave fetches its own
  // rows' span after the sequence tiles (see the end of the kernel), when a 32-column K and V tile per wave fit.
  constexpr bool OWN_FITS = Shape::W * 64 * HD * 2 <= 128 * 1024;
  const bool own_depth = OWN_FITS && waves_own_depth(a, Ld);
  const RowTilePlan plan = row_tile_plan(a, qt, BM, BN, Ld > 0 && !own_depth);
  int n_seq = plan.n_seq, n_full = plan.n_full, dep0 = plan.dep0;
  const int n_dep = plan.n_dep;
  n_seq = __builtin_amdgcn_readfirstlane(n_seq);
  n_full = __builtin_amdgcn_readfirstlane(n_full);
  dep0 = __builtin_amdgcn_readfirstlane(dep0);
  const int ntiles = __builtin_amdgcn_readfirstlane(n_seq + n_dep);

  constexpr int DMA_NOP = MODA_DMA_NOP;
  typedef AsyncTileLoader<HD, BN, NT, DMA_NOP> Loader;
  constexpr int LPT = 2 * Loader::N;
  Loader ld;
  ld.init(tid);
  typename Loader::Source srcK, srcV;
  if (a.has_seq && n_seq > 0) {
    srcK = ld.source(a.k + b * a.sk.b + hkv * a.sk.h, a.sk.t, 0, a.T, a.D);
    srcV = ld.source(a.v + b * a.sv.b + hkv * a.sv.h, a.sv.t, 0, a.T, a.Dv);
  }
  int ld_st = 0;
  auto issue = [&](int it) {
    lds_ptr Kt = smem + ld_st * 2 * BN * HD;
    if (!NODEPTH && it == n_seq) {
      srcK = ld.source(a.kd + b * a.skd.b + hkv * a.skd.h, a.skd.t, dep0, a.T * a.L, a.D);
      srcV = ld.source(a.vd + b * a.svd.b + hkv * a.svd.h, a.svd.t, dep0, a.T * a.L, a.Dv);
    }
    const int row0 = it < n_seq ? it * BN : dep0 + (it - n_seq) * BN;
    if (PARTIAL && it >= n_seq) {  // depth tile of a partially filled stream: rows through the slot mapping
      ld.load_mapped(Kt, a.kd + b * a.skd.b + hkv * a.skd.h, a.skd.t, row0, (int64_t)a.T * a.L, a.L, a.Lv, a.D);
      ld.load_mapped(Kt + BN * HD, a.vd + b * a.svd.b + hkv * a.svd.h, a.svd.t, row0, (int64_t)a.T * a.L, a.L, a.Lv,
                     a.Dv);
    } else if (WIDE) {
      const bool dep = !NODEPTH && it >= n_seq;
      const int row_end = dep ? a.T * a.L : a.T;
      ld.load(Kt, dep ? a.kd + b * a.skd.b + hkv * a.skd.h : a.k + b * a.sk.b + hkv * a.sk.h, dep ? a.skd.t : a.sk.t,
              row0, row_end, a.D);
      ld.load(Kt + BN * HD, dep ? a.vd + b * a.svd.b + hkv * a.svd.h : a.v + b * a.sv.b + hkv * a.sv.h,
              dep ? a.svd.t : a.sv.t, row0, row_end, a.Dv);
    } else {
      ld.load_from(Kt, srcK, row0);
      ld.load_from(Kt + BN * HD, srcV, row0);
    }
    ld_st = (ld_st + 1 == NST) ? 0 : ld_st + 1;
  };
  auto wait_tile = [&](int next) {
    if (DIST == 2 && next + 1 < ntiles)
      Loader::template wait_but<LPT>();
    else
      Loader::wait_all();
  };

  f32x4 dq[MB][NB];
#pragma unroll
  for (int d = 0; d < MB; d++)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) dq[d][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale * kLog2e;
  Operand16<HD> oa;
  oa.init(lane);

#pragma unroll
  for (int j = 0; j < DIST; j++)
    if (j < ntiles) issue(j);
  if (SUMS_LATE)
#pragma unroll
    for (int nb = 0; nb < NB; nb++) row_sum(nb);
  // The tile loads are issued behind the compiler's back, and a register operand it still believes pending would cost
  // a vmcnt(0) in every trip of the main loop: both kinds are waited for here, once, having travelled together.
  asm volatile("" ::: "memory");
  Loader::wait_all();
  asm volatile("" ::: "memory");
  __syncthreads();
  int c_st = 0;

  f32x4 dp_init[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) dp_init[nb] = f32x4{delta[nb], delta[nb], delta[nb], delta[nb]};
  // `nblk`: 16-column blocks of the tile (4, or 2 for a wave's own depth tiles); `scored` runs once K and V
  // have been read for the scores (V is not needed after that)
  // `emit(mb, nb, p, ds)`: called with the probabilities and the dS of every 4-column piece (the wave's own depth
  // tiles use it to hand them to the depth-gradient kernel)
  auto tile = [&](auto masked, auto nblk, lds_cptr Kc, lds_cptr Vc, int col0, const int (&lo)[NB], const int (&hi)[NB],
                  auto&& scored, auto&& emit) {
    constexpr bool MASKED = decltype(masked)::value;
    constexpr int MBLK = decltype(nblk)::value;
    f32x4 s[MBLK][NB], dp[MBLK][NB];
    mfma16_rows2<T, HD, MBLK, NB, 2>(oa, Kc, Qr, s, Vc, dOr, dp, dp_init);
    scored();
    TrPipe16<T, HD, MBLK / 2, NB, 3> kt;
    kt.prefetch(oa, Kc);
#pragma unroll
    for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        f32x4 pr;
        // a column of [lo, hi) by its distance from lo (two comparisons where the registers of the distance would spill)
        const int before = col0 + slot_base(q4) - lo[nb];
        const unsigned width = (unsigned)(hi[nb] > lo[nb] ? hi[nb] - lo[nb] : 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float p = fast_exp2(__builtin_fmaf(s[mb][nb][i], sc, -lse[nb]));
          if (MASKED && HALVES) p = (unsigned)(before + 16 * mb + i) < width ? p : 0.f;
          if (MASKED && !HALVES) {
            const int c = col0 + 16 * mb + slot_base(q4) + i;
            p = (c >= lo[nb] && c < hi[nb]) ? p : 0.f;
          }
          pr[i] = p;
          s[mb][nb][i] = p * dp[mb][nb][i];
        }
        emit(mb, nb, pr, s[mb][nb]);
      }
    i32x4 DS[MBLK / 2][NB];
#pragma unroll
    for (int ks = 0; ks < MBLK / 2; ks++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++) DS[ks][nb] = pack_slots<T>(s[2 * ks][nb], s[2 * ks + 1][nb]);
    kt.run(oa, Kc, DS, dq);
  };

  int it = 0;
  int none[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) none[nb] = 0;
  const std::integral_constant<int, 4> four{};
  const std::integral_constant<int, 2> two{};
  for (; it < n_full; it++) {
    if (it + DIST < ntiles) issue(it + DIST);
    lds_cptr Kc = smem + c_st * 2 * BN * HD;
    tile(std::false_type{}, four, Kc, Kc + BN * HD, it * BN, none, none, []() {}, [](int, int, const f32x4&, const f32x4&) {});
    c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    wait_tile(it + 1);
    __syncthreads();
  }
  // Outside chunk-visible mode (when a token's rows never straddle waves) the pass over the wave's own depth
  // columns also forms their dK and dV: see the second block below.
  constexpr bool FUSABLE = !NODEPTH && OWN_FITS && HD <= kDepthGradsInDqMaxWidth;
  bool fused_depth = false;
  if constexpr (FUSABLE) fused_depth = depth_grads_in_dq(a, HD);
  typedef WaveTileLoader<HD, DMA_NOP> Own;
  // Its private tiles: two sets of a K tile and a V tile for every wave, over the ring.  The first tile is sent for while the
  // last sequence tile is worked on, into the set that lies outside of that one's stage.
  constexpr int SET = Shape::W * 64 * HD;
  static_assert(!FUSABLE || (Shape::W == 2 && SET == 2 * BN * HD) || NST * 2 * BN * HD <= SET, "a set is a stage, or all of the ring");
  Own own;
  const uint16_t *kdp = nullptr, *vdp = nullptr;
  int c_beg = 0, c_end = 0, t_beg = 0, first_set = 0;
  bool early = false;
  auto own_tile = [&](int set) { return smem + (first_set ^ set) * SET + __builtin_amdgcn_readfirstlane(wave) * (2 * 32 * HD); };
  bool pad_k[Own::N], pad_v[Own::N];  // this lane's chunk lies past the head dim
  int rel[Own::N];                    // this lane's rows of the tile that was sent for last, from the row that `tile_row` names
  // Token `tok`, slot `slot`: those of column col0.  The rows are counted from slot 0 of the token (a full stream: from the column)
  auto tile_row = [&](int tok, int col0) { return PARTIAL ? (int64_t)tok * a.L : (int64_t)col0; };
  auto fetch = [&](int set, int col0, int tok, int slot) {
#pragma unroll
    for (int i = 0; i < Own::N; i++) {
      const int row = i * Own::RPW + own.prow;
      rel[i] = PARTIAL ? mapped_row(slot, row, a.L, a.Lv) : row;
      rel[i] = col0 + row < c_end ? rel[i] : -1;
    }
    const int64_t row0 = tile_row(tok, col0), rows = (int64_t)a.T * a.L;
    const uint32_t sk = (uint32_t)a.skd.t * 2u, sv = (uint32_t)a.svd.t * 2u;
    lds_ptr Kt = own_tile(set);
    own.fetch_rows(Kt, kdp + row0 * a.skd.t, sk, mapped_bytes(row0, rows, sk), rel, pad_k);
    own.fetch_rows(Kt + 32 * HD, vdp + row0 * a.svd.t, sv, mapped_bytes(row0, rows, sv), rel, pad_v);
  };
  auto enter_depth = [&]() {
    const int rw0 = qt * BM + __builtin_amdgcn_readfirstlane(wave) * WR;
    if (rw0 >= a.Tq) return;
    const DepthSpan span = own_depth_span(a, rw0, WR);
    c_beg = __builtin_amdgcn_readfirstlane(span.c_beg);
    c_end = __builtin_amdgcn_readfirstlane(span.c_end);
    t_beg = __builtin_amdgcn_readfirstlane(span.t_beg);
    kdp = a.kd + b * a.skd.b + hkv * a.skd.h;
    vdp = a.vd + b * a.svd.b + hkv * a.svd.h;
    own.init(lane);
#pragma unroll
    for (int i = 0; i < Own::N; i++) {
      pad_k[i] = own.chunk(i) * 8 >= a.D;
      pad_v[i] = own.chunk(i) * 8 >= a.Dv;
    }
    if (c_beg < c_end) fetch(0, c_beg, t_beg, 0);
  };
  for (; it < ntiles; it++) {
    if (it + DIST < ntiles) issue(it + DIST);
    if (FUSABLE && fused_depth && it + 1 == ntiles) {
      first_set = dq_first_private_set(Shape::W, c_st);
      enter_depth();
      early = true;
    }
    const bool dep = !NODEPTH && it >= n_seq;
    const int col0 = dep ? dep0 + (it - n_seq) * BN : it * BN;
    int lo[NB], hi[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      lo[nb] = dep ? dlo[nb] : 0;
      hi[nb] = dep ? dhi[nb] : shi[nb];
    }
    lds_cptr Kc = smem + c_st * 2 * BN * HD;
    auto part = [&](auto nblk, lds_cptr Kp, int c) {
      constexpr int COLS = 16 * decltype(nblk)::value;
      bool touches = false;
#pragma unroll
      for (int nb = 0; nb < NB; nb++) touches = touches || ((hi[nb] > c) && (lo[nb] < c + COLS) && (hi[nb] > lo[nb]));
      if (__any(touches)) tile(std::true_type{}, nblk, Kp, Kp + BN * HD, c, lo, hi, []() {}, [](int, int, const f32x4&, const f32x4&) {});
    };
    if constexpr (HALVES) {  // by halves: the last tile of a sequence is as often as not seen by no row beyond its first half
#pragma unroll 1
      for (int c = col0; c < col0 + BN; c += 32, Kc += 32 * HD) part(two, Kc, c);
    } else {
      part(four, Kc, col0);
    }
    c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    if (it + 1 < ntiles) wait_tile(it + 1);
    __syncthreads();
  }

  if (own_depth && !fused_depth) {
    // The wave's own depth columns, 32 at a time through a wave-private K tile and V tile cut out of the ring
    // (no workgroup barrier after the one that retires the ring).  The next V tile is fetched as soon as the
    // scores are out, the next K tile once dQ has its share.
    __syncthreads();
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    lds_ptr Kt = smem + wv * (2 * 32 * HD), Vt = Kt + 32 * HD;
    const int rw0 = qt * BM + wv * WR;
    if (rw0 < a.Tq) {
      const DepthSpan span = own_depth_span(a, rw0, WR);
      const int c_beg = __builtin_amdgcn_readfirstlane(span.c_beg);
      const int c_end = __builtin_amdgcn_readfirstlane(span.c_end);
      const int nh = (c_end - c_beg + 31) / 32;
      const uint16_t* kdp = a.kd + b * a.skd.b + hkv * a.skd.h;
      const uint16_t* vdp = a.vd + b * a.svd.b + hkv * a.svd.h;
      Own own;
      own.init(lane);
      // rows [col0, col0 + 32) of the span (short at its end) into a private tile; d: the tensor's head dim
      auto fetch = [&](lds_ptr tile, const uint16_t* slice, int64_t stride, int col0, int d) {
        const int nrows = min(32, c_end - col0);
        if (PARTIAL)
          own.fetch_mapped(tile, slice, stride, col0, nrows, (int64_t)a.T * a.L, a.L, a.Lv, d);
        else
          own.fetch(tile, slice, stride, col0, nrows, d);
      };
      fetch(Kt, kdp, a.skd.t, c_beg, a.D);
      fetch(Vt, vdp, a.svd.t, c_beg, a.Dv);
      // where the depth-gradient kernel takes P and dS from here: this lane's rows of the two arrays
      const bool hand_over = a.depth_p != nullptr;
      uint16_t *hp[NB], *hds[NB];
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const int r = rw0 + 16 * nb + n, t = r / a.Gf;  // slot l of row r: element l * Gf + (r - t * Gf) of token t's block
        const int64_t at = (((int64_t)b * a.Hq + hq) * (VARLEN ? a.delta_pitch : a.Tq) + (int64_t)t * a.Gf) * a.Lv + (r - t * a.Gf);
        hp[nb] = a.depth_p + at;
        hds[nb] = a.depth_ds + at;
      }
      for (int j = 0; j < nh; j++) {
        const int col0 = c_beg + 32 * j;
        const bool more = j + 1 < nh;
        Own::template wait_but<0>();
        tile(std::true_type{}, two, Kt, Vt, col0, dlo, dhi,
             [&]() {
               Own::reads_done();
               if (more) fetch(Vt, vdp, a.svd.t, col0 + 32, a.Dv);
             },
             [&](int mb, int nb, const f32x4& p, const f32x4& ds) {
               if (!hand_over) return;
               // rounded as the matrix products take them; slot of column c within its row: c - dlo
               const int w0 = pack2<T>(p[0], p[1]), w1 = pack2<T>(p[2], p[3]);
               const int x0 = pack2<T>(ds[0], ds[1]), x1 = pack2<T>(ds[2], ds[3]);
#pragma unroll
               for (int i = 0; i < 4; i++) {
                 const int c = col0 + 16 * mb + slot_base(q4) + i;
                 if (c >= dlo[nb] && c < dhi[nb]) {
                   const int pw = (i < 2) ? w0 : w1, dw = (i < 2) ? x0 : x1;
                   hp[nb][(c - dlo[nb]) * a.Gf] = (uint16_t)((i & 1) ? ((unsigned)pw >> 16) : ((unsigned)pw & 0xffffu));
                   hds[nb][(c - dlo[nb]) * a.Gf] = (uint16_t)((i & 1) ? ((unsigned)dw >> 16) : ((unsigned)dw & 0xffffu));
                 }
               }
             });
        Own::reads_done();
        if (more) fetch(Kt, kdp, a.skd.t, col0 + 32, a.D);
      }
    }
  }

  // The wave's own depth columns when no other wave sees them (moda_v14.py:1251-1454, fda_v12.py:646-860 for
  // their dK/dV): the products run the other way round here, S = Q Kd^T with the query rows on the accumulator
  // registers (rows 4q + i of each 16-row block) and the depth column on the lane.  P and dS of the wave's 32 rows,
  // rounded and packed, then ARE the operands (summation index = query row) of dVd^T = dO^T P and
  // dKd^T = Q^T dS: one matrix instruction per 16 columns x 16 head-dim elements, nothing to accumulate across
  // tiles.  Q^T and dO^T in that slot order are read once, through the private tiles before the first fetch.
  // dQ needs dS with the columns as summation index: the rounded dS block crosses over through a small LDS block
  // of the wave.
  if constexpr (FUSABLE) {
    if (fused_depth) {
      static_assert(NB == 2, "the wave's 32 query rows are the 32 summation slots of one matrix instruction");
      if (!early) enter_depth();  // (every ring tile ends with a barrier)
      const int wv = __builtin_amdgcn_readfirstlane(wave);
      // behind the two sets the 32 x 32 dS block
      lds_ptr stage = smem + 2 * SET + wv * (16 * HD);
      const int rw0 = qt * BM + wv * WR;
      if (rw0 < a.Tq) {
        lds_ptr Kt = own_tile(1), Vt = Kt + 32 * HD;  // (the first tile is on its way to the other set)
        // Query row 16*nb + n goes to the tile row its lane reads as a row operand, slot_base(n >> 2) + (n & 3):
        // the transposed read then delivers rows 4q + j and 16 + 4q + j as lane group q's eight summation slots,
        // the order of the packed accumulators.
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
          for (int ks = 0; ks < KS; ks++) {
            *reinterpret_cast<MODA_LDS i32x4*>(Kt + oa.row[ks] + 16 * nb * HD) = Qr[nb][ks];
            *reinterpret_cast<MODA_LDS i32x4*>(Vt + oa.row[ks] + 16 * nb * HD) = dOr[nb][ks];
          }
        Own::reads_done();  // (the counter covers LDS writes as well)
        i32x4 QT[MB], dOT[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          QT[mb] = oa.tr_operand(Kt, 0, mb);
          dOT[mb] = oa.tr_operand(Vt, 0, mb);
        }
        Own::reads_done();
        // per accumulator register: base-2 LSE and minus delta of query row 16*nb + 4*q4 + i, from the lanes that
        // hold those rows (lane n of the first sixteen holds row 16*nb + n; rows past the end carry zeros)
        f32x4 lse4[NB], del4[NB];
        const int rq = rw0 + 4 * q4;
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            lse4[nb][i] = __shfl(lse[nb], 4 * q4 + i, 64);
            del4[nb][i] = __shfl(delta[nb], 4 * q4 + i, 64);
          }
        const int gshift = __builtin_ctz(a.Gf);  // Gf divides 32: a power of two
        const int nh = (c_end - c_beg + 31) / 32;
        // Token of the query row on accumulator register i of block nb: the first register's and i >> gshift more (rows past the end
        // belong to tokens that no column has).  Every register counts here: spilled ones, 11 in fp16, cost a launch that streams
        // from memory 5 %.
        int row_token[NB];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) row_token[nb] = (rq + 16 * nb) >> gshift;
        const uint16_t* dkdp = a.dkd + b * a.sdkd.b + hkv * a.sdkd.h;
        const uint16_t* dvdp = a.dvd + b * a.sdvd.b + hkv * a.sdvd.h;
        const int lrow = slot_base(n >> 2) + (n & 3);  // tile row (of a 16-row block) whose column this lane holds
        // The rounded dS block crosses over through `stage`: per 16 columns and 16 query rows, column by column in lane order,
        // four rows (8 bytes) a piece; columns 8 .. 15 have their two halves swapped, which spreads the pieces that are written
        // together over all banks.  The transposed read hands lane group q the columns slot_base(q) .. + 3 of each block.
        const int xs_put = n * 16 + 4 * (q4 ^ ((n >> 3) << 1)), xs_col = 4 * q4 + (n >> 2), xs_get = xs_col * 16 + 4 * ((n & 3) ^ ((xs_col >> 3) << 1));
        int tok = t_beg, slot = 0;  // of the tile's first column
        // Tile j: wait for its rows, send for tile j + 1 (other set), scores, dS and dQ; then its gradient rows, through the
        // tile's own K and V blocks, which nobody reads any more: the accumulators hold 8-byte pieces of 16 different rows per
        // register, which the memory pipeline would take as 16 partial lines per store; written to LDS and read back by rows,
        // every store covers whole rows.  The wave's memory counter covers loads and stores alike: the wait for the next
        // tile's rows leaves this tile's eight stores, younger than them, on their way.  Such a launch is bound by what a wave has to
        // issue, one thing after the other (six slots of twelve, 64 x 197 tokens of four rows: 43 k cycles): with 16 rows staged
        // at a time, guarded 64-bit addresses and dS crossing in 2-byte pieces a backward pass over the stream's layers took
        // 27.8 us a dQ launch, now 24.9; vision layers (64 x 197, six heads, twelve slots) 190 -> 184 us a step.
        for (int j = 0; j < nh; j++) {
          const int col0 = c_beg + 32 * j;
          lds_ptr Kc = own_tile(j & 1), Vc = Kc + 32 * HD;
          const SlotStep ahead = slot_step(slot, 32, a.Lv);
          const int next_tok = tok + __builtin_amdgcn_readfirstlane(ahead.tokens), next_slot = __builtin_amdgcn_readfirstlane(ahead.slot);
          if (j == 0)
            Own::template wait_but<0>();
          else
            Own::template wait_but<2 * Own::N>();
          int grow[Own::N];  // this lane's rows of the tile
#pragma unroll
          for (int i = 0; i < Own::N; i++) grow[i] = rel[i];
          auto off_k = [&](int i) { return own.row_offset(i, grow[i], (int)a.sdkd.t * 2, pad_k[i]); };
          auto off_v = [&](int i) { return own.row_offset(i, grow[i], (int)a.sdvd.t * 2, pad_v[i]); };
          const int64_t row0 = tile_row(tok, col0);
          const RowBuffer dk_rows(dkdp + row0 * a.sdkd.t, kPadOffset), dv_rows(dvdp + row0 * a.sdvd.t, kPadOffset);
          if (j + 1 < nh) fetch((j + 1) & 1, col0 + 32, next_tok, next_slot);
          f32x4 s[2][NB], dp[2][NB];
          mfma16_rows2<T, HD, 2, NB, 2, true>(oa, Kc, Qr, s, Vc, dOr, dp, del4);
          // Accumulating: what the gradient rows hold, sent for once the scores are out of the registers (where it is added,
          // every row would stand still for a trip to memory)
          i32x4 old_k[Own::N], old_v[Own::N], PA[2], DSA[2];
          if (a.accum_depth) {
#pragma unroll
            for (int i = 0; i < Own::N; i++) {
              old_v[i] = dv_rows.load(off_v(i));
              old_k[i] = dk_rows.load(off_k(i));
            }
          }
#pragma unroll
          for (int cb = 0; cb < 2; cb++) {
            const int tokc = col0 + 16 * cb + lrow < c_end ? tok + slot_step(slot, 16 * cb + lrow, a.Lv).tokens : -2;
            f32x4 p[NB], ds[NB];
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
              for (int i = 0; i < 4; i++) {
                float pv = fast_exp2(__builtin_fmaf(s[cb][nb][i], sc, -lse4[nb][i]));
                pv = tokc - row_token[nb] == (i >> gshift) ? pv : 0.f;
                p[nb][i] = pv;
                ds[nb][i] = pv * dp[cb][nb][i];
              }
            PA[cb] = pack_slots<T>(p[0], p[1]);
            DSA[cb] = pack_slots<T>(ds[0], ds[1]);
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
              *reinterpret_cast<MODA_LDS i32x2*>(stage + (2 * cb + nb) * 256 + xs_put) = i32x2{DSA[cb][2 * nb], DSA[cb][2 * nb + 1]};
          }
          Own::reads_done();  // (the counter covers LDS writes as well)
          i32x4 DS[1][NB];
#pragma unroll
          for (int nb = 0; nb < NB; nb++) {
            const i32x2 lo = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((MODA_LDS s16x4*)(stage + nb * 256 + xs_get)));
            const i32x2 hi = __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((MODA_LDS s16x4*)(stage + (2 + nb) * 256 + xs_get)));
            DS[0][nb] = i32x4{lo[0], lo[1], hi[0], hi[1]};
          }
          TrPipe16<T, HD, 1, NB, 3> kt;
          kt.prefetch(oa, Kc);
          kt.run(oa, Kc, DS, dq);
          Own::reads_done();
          auto put = [&](lds_ptr block, int cb, int mb, const f32x4& x, float mul) {
            i32x2 w;
            w[0] = pack2<T>(x[0] * mul, x[1] * mul);
            w[1] = pack2<T>(x[2] * mul, x[3] * mul);
            *reinterpret_cast<MODA_LDS i32x2*>(block + 16 * cb * HD + Tile<HD>::off(lrow, 2 * mb + (q4 >> 1)) + 4 * (q4 & 1)) = w;
          };
          const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int cb = 0; cb < 2; cb++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
              put(Vc, cb, mb, mfma16<T>(dOT[mb], PA[cb], z), 1.f);
              put(Kc, cb, mb, mfma16<T>(QT[mb], DSA[cb], z), a.scale);
            }
          Own::reads_done();
          auto flush = [&](lds_ptr block, const RowBuffer& rows, auto&& off, const i32x4 (&old)[Own::N]) {
#pragma unroll
            for (int i = 0; i < Own::N; i++) {
              i32x4 val = *reinterpret_cast<MODA_LDS const i32x4*>(block + i * 512 + lane * 8);
              if (a.accum_depth) {  // add to what the row holds (this lane is the only writer of its 16 bytes)
#pragma unroll
                for (int w = 0; w < 4; w++) {
                  float x0, x1, y0, y1;
                  unpack2<T>(val[w], x0, x1);
                  unpack2<T>(old[i][w], y0, y1);
                  val[w] = pack2<T>(x0 + y0, x1 + y1);
                }
              }
              rows.template store<true>(val, off(i));  // next read by another launch
            }
          };
          flush(Vc, dv_rows, off_v, old_v);
          flush(Kc, dk_rows, off_k, old_k);
          Own::reads_done();  // this set may be loaded over
          tok = next_tok;
          slot = next_slot;
        }
      }
    }
  }

#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const int r = qt * BM + wave * WR + 16 * nb + n;
    if (r < a.Tq) {
      uint16_t* op = a.dq + b * a.sdq.b + hq * a.sdq.h + (int64_t)r * a.sdq.t;
#pragma unroll
      for (int d = 0; d < MB; d++) {
        i32x2 w;
        w[0] = pack2<T>(dq[d][nb][0] * a.scale, dq[d][nb][1] * a.scale);
        w[1] = pack2<T>(dq[d][nb][2] * a.scale, dq[d][nb][3] * a.scale);
        if (16 * d + 4 * q4 < a.D) {
          i32x2* dst = reinterpret_cast<i32x2*>(op + 16 * d + 4 * q4);
          // the narrow tiles serve HBM-bound shapes whose depth stream can stay in the memory-side cache between
          // launches if results written once do not displace it
          if (HD <= 64)
            __builtin_nontemporal_store(w, dst);
          else
            *dst = w;
        }
      }
    }
  }
}

// LDS of a workgroup: the ring, or one 32-column K tile and V tile per wave for the waves' own depth columns
// ... and, where the kernel forms the depth gradients, a second set of those and a 32 x 32 block per wave (16 rows of HD) through
// which dS crosses over
template <int HD, typename Shape, int ADDR>
constexpr size_t dq_lds() {
  constexpr size_t ring = (size_t)Shape::NST * 2 * 64 * HD * sizeof(uint16_t),
                   own = (size_t)Shape::W * (HD <= kDepthGradsInDqMaxWidth ? 2 * 64 + 16 : 64) * HD * sizeof(uint16_t);
  return (ADDR & 4) == 0 && (size_t)Shape::W * 64 * HD * sizeof(uint16_t) <= 128 * 1024 ? (ring > own ? ring : own) : ring;
}

}  // namespace moda
