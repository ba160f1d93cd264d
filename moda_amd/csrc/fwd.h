// Forward kernel of the tiles up to 128 wide: the body (fwd_kernel.hip has what it computes and how it is laid out).
#pragma once
#include <type_traits>

#include "geometry.h"
#include "kargs.h"
#include "tile.h"
#include "tuning.h"

namespace moda {

// ADDR bit 0: a (batch, head) slice is wider than 2 GiB (descriptors anchored per tile instead of 32-bit
// offsets inside the slice); bit 1: packed variable-length batch; bit 2: no depth stream; bit 3: partially filled
// depth stream (only Lv of a token's L slots hold data: depth tiles are loaded through the slot mapping)
// On the 64-wide tiles the registers of three waves per SIMD are enough (168, no spills).
// The body is a kernel of its own, or (MODA_SIDE_BY_SIDE, attend_tail_kernel.hip) a function that works on the query tile `place`
// and hands the rows to `out(row of the tile, chunk, half, 4 values)` instead of memory, every row of the tile, once the whole
// workgroup has done reading its `smem`.
template <typename T, int HD, typename Shape, int ADDR
#ifdef MODA_SIDE_BY_SIDE
          , typename Out>
__device__ __forceinline__ void fwd_body(const KArgs& a_in, const RowPlace& place, lds_ptr smem, lds_ptr apart_k, lds_ptr apart_v, Out&& out) {
#else
          >
__global__ __launch_bounds__(64 * Shape::W, HD <= 64 ? 3 : 2) void fwd_kernel(const KArgs a_in) {
#endif
#ifdef MODA_SIDE_BY_SIDE
  constexpr int WORKING = Shape::WORKING;
#else
  constexpr int WORKING = Shape::W;
#endif
  constexpr int BM = 32 * WORKING, BN = 64, KK = HD / 16, DB = HD / 32, NT = 64 * Shape::W, NST = Shape::NST,
                DIST = Shape::DIST;
  constexpr bool PP = Shape::PP;
  static_assert(NST >= DIST + 1 + (PP ? 1 : 0) && DIST >= 1 && DIST <= 3,
                "ring must hold the tile in use, the tiles in flight and (ping-pong) the previous tile");
  static_assert(2 * NST >= Shape::W, "the ring must be large enough for one 32-column K tile and V tile per wave");
#ifndef MODA_SIDE_BY_SIDE
  extern __shared__ __align__(16) unsigned char smem_raw[];
  lds_ptr smem = (lds_ptr)smem_raw;  // ring stage st: K tile at smem + st * 2*BN*HD, V tile right behind it
#endif

#ifdef MODA_SIDE_BY_SIDE
  const int tid = (int)threadIdx.x % (64 * Shape::W);  // (half of the workgroup may be at another head: as many barriers there)
#else
  const int tid = threadIdx.x;
#endif
  const int lane = tid & 63, wave = tid >> 6, n = lane & 31, g = lane >> 5;
  constexpr bool WIDE = (ADDR & 1) != 0, VARLEN = (ADDR & 2) != 0;
  // bit 2: launched without a depth stream (the plain and sequence-only calls): the depth code is compiled out,
  // so that it cannot disturb the register allocation of their main loop
  constexpr bool NODEPTH = (ADDR & 4) != 0, PARTIAL = (ADDR & 8) != 0;
  static_assert(!(NODEPTH && PARTIAL), "a partially filled depth stream is a depth stream");
#ifndef MODA_SIDE_BY_SIDE
  const RowPlace place = row_place<VARLEN>(a_in, (int)blockIdx.x, BM);
  if (VARLEN && !place.active) return;
#endif
  int b = place.b;
  const int hq = place.hq, hkv = hq / a_in.hdiv, qt = place.qt;
  SeqArgs<VARLEN> seq(a_in, b, place.t0, place.T);
  const KArgs& a = seq.a;
  const int Ld = NODEPTH ? 0 : a.L;  // depth slots per token
  const bool idle = WORKING < Shape::W && __builtin_amdgcn_readfirstlane(wave) >= WORKING;  // only loads tiles
  const int r = qt * BM + wave * 32 + n;
  const bool valid = r < a.Tq && !idle;
  const int t = r / a.Gf;

  i32x4 Qr[KK];
  {
    const uint16_t* qp = a.q + b * a.sq.b + hq * a.sq.h + (int64_t)r * a.sq.t + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
      i32x4 z = {0, 0, 0, 0};
      Qr[kk] = (valid && 16 * kk + 8 * g < a.D) ? *reinterpret_cast<const i32x4*>(qp + 16 * kk) : z;
    }
  }

  // per-row visible column intervals [lo, hi) for the two phases
  const RowVis vis = row_visibility(a, r, Ld);
  const int shi = vis.shi, dlo = vis.dlo, dhi = vis.dhi;
  // Depth columns a wave alone can see are not streamed through the workgroup's ring: each wave fetches its own
  // rows' span after the sequence tiles (see the end of the kernel).
  const bool own_depth = waves_own_depth(a, Ld);
  const RowTilePlan plan = row_tile_plan(a, qt, BM, BN, Ld > 0 && !own_depth);
  int n_seq = plan.n_seq, n_full = plan.n_full, dep0 = plan.dep0;
  const int n_dep = plan.n_dep;
  // wave-uniform by construction, but computed with vector divisions: the explicit hint keeps the
  // loop control in scalar registers
  n_seq = __builtin_amdgcn_readfirstlane(n_seq);
  n_full = __builtin_amdgcn_readfirstlane(n_full);
  dep0 = __builtin_amdgcn_readfirstlane(dep0);
  const int ntiles = __builtin_amdgcn_readfirstlane(n_seq + n_dep);

  typedef AsyncTileLoader<HD, BN, NT> Loader;
  constexpr int LPT = 2 * Loader::N;  // vector-memory loads one wave issues per tile (K + V)
  Loader ld;
  ld.init(tid);
  // the two sources being streamed: sequence K/V first, swapped for the depth K/V when the
  // producer reaches the first depth tile
  typename Loader::Source srcK, srcV;
  if (a.has_seq && n_seq > 0) {
    srcK = ld.source(a.k + b * a.sk.b + hkv * a.sk.h, a.sk.t, 0, a.T, a.D);
    srcV = ld.source(a.v + b * a.sv.b + hkv * a.sv.h, a.sv.t, 0, a.T, a.Dv);
  }
  int ld_st = 0;  // ring stage the next issued tile goes to
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
    } else if (WIDE) {  // some slice spans more than 2 GiB: a descriptor anchored at this tile
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
  // wait until tile `next` has landed; tiles next+1 .. next+DIST-1 may still be in flight
  auto wait_tile = [&](int next) {
    if (DIST == 3 && next + 2 < ntiles)
      Loader::template wait_but<2 * LPT>();
    else if (DIST >= 2 && next + 1 < ntiles)
      Loader::template wait_but<LPT>();
    else
      Loader::wait_all();
  };

  f32x16 o[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[d][i] = 0.f;
  float m = kNegInf, l = 0.f;
  const float sc = a.scale * kLog2e;
  OperandAddr<HD> oa;
  oa.init(lane);

#ifndef MODA_SIDE_BY_SIDE
#pragma unroll
  for (int j = 0; j < DIST; j++)
    if (j < ntiles) issue(j);
  // The tile loads are issued behind the compiler's back, and a register operand it still believes pending would cost
  // a vmcnt(0) in every trip of the main loop: both kinds are waited for here, once, having travelled together.
  asm volatile("" ::: "memory");
  Loader::wait_all();
  asm volatile("" ::: "memory");
  __syncthreads();
#endif
  int c_st = 0;  // ring stage of the tile being consumed

  // One column tile in two halves.  front: S^T = K Q^T and the online softmax, leaving the rounded
  // probabilities in P; back: O^T += V^T P^T.
  i32x4 P[4];
  TrPipe<T, HD, 4, 2> pv;
  const std::integral_constant<int, 2> two{};
  const std::integral_constant<int, 1> one{};
  auto front = [&](auto masked, auto nblk, lds_cptr Kc, int col0, int lo, int hi, auto&& after_scores) {
    constexpr bool MASKED = decltype(masked)::value;
    constexpr int NBLK = decltype(nblk)::value;  // 32-column blocks of the tile
    f32x16 s[NBLK];
    mfma_rows<T, HD, NBLK, 4>(oa, Kc, Qr, s);
    after_scores();
    // whether the row sees register i of block bb, a column of [lo, hi): by its distance from lo (0 without depth)
    const int before = col0 + 4 * g - lo;
    const unsigned width = (unsigned)(hi > lo ? hi - lo : 0);
    auto sees = [&](int bb, int i) {
      return NODEPTH ? col0 + 32 * bb + acc_row(i, g) < hi : (unsigned)(before + 32 * bb + acc_row(i, 0)) < width;
    };
    // row maximum of the raw scores (scale > 0, so it commutes with the max)
    float mx = kNegInf;
#pragma unroll
    for (int bb = 0; bb < NBLK; bb++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        if (MASKED) {
          mx = fmaxf(mx, sees(bb, i) ? s[bb][i] : kNegInf);
        } else {
          mx = fmaxf(mx, s[bb][i]);
        }
      }
    mx = pair_max(mx) * sc;
    // The exponent reference m only moves when some row's maximum outgrows it by more than 2^8:
    // p stays <= 256, exact in fp32 accumulation and harmless in the 16-bit P, and the
    // rescale of O is skipped on almost every tile.
    if (__any(mx > m + 8.f)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = fast_exp2(m - ((m_new == kNegInf) ? 0.f : m_new));
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] *= alpha;
    }
    const float neg_m = (m == kNegInf) ? 0.f : -m;
    float rs0 = 0.f, rs1 = 0.f;  // fp32 row sum of the unrounded probabilities, as the reference keeps it
#pragma unroll
    for (int bb = 0; bb < NBLK; bb++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        float p = fast_exp2(__builtin_fmaf(s[bb][i], sc, neg_m));
        if (MASKED) p = sees(bb, i) ? p : 0.f;
        s[bb][i] = p;
        if (i & 1)
          rs1 += p;
        else
          rs0 += p;
      }
#pragma unroll
    for (int ks = 0; ks < 2 * NBLK; ks++) P[ks] = pack8<T>(s[ks >> 1], (ks & 1) * 8);
    l += pair_sum(rs0 + rs1);
  };
  // the whole tile at once: the first V^T operands start travelling while the softmax runs
  auto tile = [&](auto masked, lds_cptr Kc, lds_cptr Vc, int col0, int lo, int hi) {
    front(masked, two, Kc, col0, lo, hi, [&]() { pv.prefetch(oa, Vc); });
    pv.run(oa, Vc, P, o);
  };
  auto back = [&](lds_cptr Vc) {
    pv.prefetch(oa, Vc);
    pv.run(oa, Vc, P, o);
  };
  // 32 columns, masked
  auto half_tile = [&](lds_cptr Kc, lds_cptr Vc, int col0, int lo, int hi, auto&& after_scores) {
    TrPipe<T, HD, 2, 2> pv1;
    front(std::true_type{}, one, Kc, col0, lo, hi, [&]() {
      after_scores();
      pv1.prefetch(oa, Vc);
    });
    const i32x4 P1[2] = {P[0], P[1]};
    pv1.run(oa, Vc, P1, o);
  };
  auto stage_k = [&](int st) { return smem + st * 2 * BN * HD; };

  // The wave's own depth columns, 32 at a time through wave-private K and V tiles cut out of the ring.  EARLY: the first
  // ones travel while the last sequence tile is worked on, into the ring stage that is free by then.  Two waves have room
  // for two whole sets, one in each stage, and fetch a tile ahead all the way; four for K in one stage and V in the other.
  // A short launch is bound by what one wave has to do, one thing after the other: 64 x 197 tokens of four rows, eleven of
  // twelve slots filled, 35.5 k cycles a wave with every private tile waited for and 13.7 k of them in this pass; now 29.1 k
  // and 7.0 k, the launch 16.5 -> 13.9 us (six slots 14.1 -> 12.5).
  // APART (MODA_SIDE_BY_SIDE): the first set lies beside the ring and is sent for before the first sequence tile is worked on, the
  // second one lies over the ring.
  constexpr bool APART = Shape::APART, EARLY = !NODEPTH && !PP && (NST == 2 || APART) && HD <= 64, TWO_SETS = EARLY && (Shape::W <= 2 || APART);
  typedef WaveTileLoader<HD> Own;
  Own own;
  const uint16_t *kdp = nullptr, *vdp = nullptr;
  int c_beg = 0, c_end = 0, tok = 0, slot = 0;  // the span; token and slot of the next tile to be fetched
  int first_set = 0;
  bool early = false;
  auto enter_depth = [&]() {
    const int rw0 = qt * BM + __builtin_amdgcn_readfirstlane(wave) * 32;
    if (rw0 >= a.Tq || idle) return;
    const DepthSpan span = own_depth_span(a, rw0, 32);
    c_beg = __builtin_amdgcn_readfirstlane(span.c_beg);
    c_end = __builtin_amdgcn_readfirstlane(span.c_end);
    tok = __builtin_amdgcn_readfirstlane(span.t_beg);
    kdp = a.kd + b * a.skd.b + hkv * a.skd.h;
    vdp = a.vd + b * a.svd.b + hkv * a.svd.h;
    own.init(lane);
  };
  // rows [col0, col0 + 32) of the span (short at its end) into a private tile; d: the tensor's head dim
  auto fetch = [&](lds_ptr tile, const uint16_t* slice, int64_t stride, int col0, int d) {
    const int nrows = min(32, c_end - col0);
    if (PARTIAL)
      own.fetch_slots(tile, slice, stride, tok, slot, nrows, (int64_t)a.T * a.L, a.L, a.Lv, d);
    else
      own.fetch(tile, slice, stride, col0, nrows, d);
  };
  auto next_columns = [&]() {
    if (!PARTIAL) return;
    const SlotStep s = slot_step(slot, 32, a.Lv);
    tok += __builtin_amdgcn_readfirstlane(s.tokens);
    slot = __builtin_amdgcn_readfirstlane(s.slot);
  };
  auto own_tile = [&](int set) {
    const int wv = __builtin_amdgcn_readfirstlane(wave);
#ifdef MODA_SIDE_BY_SIDE
    return set == 0 ? apart_k + wv * (32 * HD) : smem + wv * (2 * 32 * HD);
#else
    return !EARLY ? smem + wv * (2 * 32 * HD) : stage_k(first_set ^ set) + wv * (TWO_SETS ? 2 * 32 * HD : 32 * HD);
#endif
  };
  auto own_v = [&](int set) {  // its V tile, with two sets
#ifdef MODA_SIDE_BY_SIDE
    if (set == 0) return apart_v + __builtin_amdgcn_readfirstlane(wave) * (32 * HD);
#endif
    return own_tile(set) + 32 * HD;
  };
  auto fetch_early = [&]() {
    fetch(own_tile(0), kdp, a.skd.t, c_beg, a.D);
    if (TWO_SETS) {
      fetch(own_v(0), vdp, a.svd.t, c_beg, a.Dv);
      next_columns();
    }
  };
#ifdef MODA_SIDE_BY_SIDE
  // First tiles of the ring and of the wave, and whatever else is on its way by now, travel together.
  static_assert(APART, "a body whose caller has other uses for the ring");
#pragma unroll
  for (int j = 0; j < DIST; j++)
    if (j < ntiles) issue(j);
  if (EARLY && own_depth) {
    enter_depth();
    if (c_beg < c_end) fetch_early();
    early = true;
  }
  asm volatile("" ::: "memory");
  Loader::wait_all();
  asm volatile("" ::: "memory");
  __syncthreads();
#endif

  // Ping-pong: the two waves of a SIMD (wave w and w + W/2) would otherwise run the same phase at the
  // same time -- matrix pipe contended during the MFMA phases, idle during both softmaxes.  The upper
  // half of the workgroup therefore runs half a tile behind: between two barriers it first finishes the
  // previous tile (V product), then does scores and softmax of the current one, so its softmax overlaps
  // the lower half's V product and its V product the lower half's scores.  The previous tile's V must
  // survive one more barrier interval, hence the extra ring stage.
  const bool late = PP && __builtin_amdgcn_readfirstlane(wave) >= Shape::W / 2;
  int it = 0;
  if (idle) {
    for (; it < ntiles; it++) {
      if (it + DIST < ntiles) issue(it + DIST);
      wait_tile(it + 1);
      __syncthreads();
    }
  } else if (!late) {
    // phase 1: tiles fully visible to every row -- no masks, no visibility tests.  The loop is unrolled
    // over the ring stages so that each copy reads its tile at a compile-time LDS offset (the stage
    // offset then rides in the instructions' immediate field instead of costing an address add per
    // operand read); the remainder runs the same body with the stage in a register.
    auto full_tile = [&](lds_cptr Kc) {
      if (it + DIST < ntiles) issue(it + DIST);
      tile(std::false_type{}, Kc, Kc + BN * HD, it * BN, 0, 0);
      wait_tile(it + 1);
      __syncthreads();
      it++;
    };
    for (; it + NST <= n_full;) {
      full_tile(smem);
      full_tile(smem + 1 * 2 * BN * HD);
      if (NST > 2) full_tile(smem + 2 * 2 * BN * HD);
      if (NST > 3) full_tile(smem + 3 * 2 * BN * HD);
    }
    c_st = 0;
    for (; it < n_full;) {
      full_tile(stage_k(c_st));
      c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    }
    // phase 2: boundary sequence tiles and depth tiles
    for (; it < ntiles; it++) {
      if (it + DIST < ntiles) issue(it + DIST);
      if (EARLY && !APART && own_depth && it + 1 == ntiles) {
        first_set = fwd_first_private_set(c_st);
        enter_depth();
        if (c_beg < c_end) fetch_early();
        early = true;
      }
      const bool dep = !NODEPTH && it >= n_seq;
      const int col0 = dep ? dep0 + (it - n_seq) * BN : it * BN;
      const int lo = dep ? dlo : 0;
      const int hi = dep ? dhi : shi;
      lds_cptr Kc = stage_k(c_st);
      const auto seen = [&](int c, int cols) { return __any((hi > c) && (lo < c + cols) && (hi > lo)); };
      if (HD <= 64 && !NODEPTH && seen(col0, 32) != seen(col0 + 32, 32)) {
        // No row of the wave sees the other half, as in every second last tile of a sequence: 32 columns give the bits of the whole tile,
        // which takes one maximum over all of them.  Serving twelve blocks of 64 x 197 tokens, five columns in the last tile: 566 us
        // with whole tiles, 559 so; one such layer of six heads 199 both.  (Without depth the whole tile is as fast: 13.1 us by halves and
        // 12.9.)
        const int half = seen(col0, 32) ? 0 : 32;
        half_tile(Kc + half * HD, Kc + (BN + half) * HD, col0 + half, lo, hi, []() {});
      } else if (seen(col0, BN)) {
        tile(std::true_type{}, Kc, Kc + BN * HD, col0, lo, hi);
      }
      c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
      if (it + 1 < ntiles) wait_tile(it + 1);
      __syncthreads();
    }
  } else {
    // the late half: [V product of the previous tile] [scores + softmax of this tile] [barrier]
    if (n_full > 0) {  // first tile: nothing to finish yet
      if (DIST < ntiles) issue(DIST);
      front(std::false_type{}, two, smem, 0, 0, 0, []() {});
      wait_tile(1);
      __syncthreads();
      it = 1;
    }
    // `Vp`: V tile of the previous tile, `Kc`: K tile of this one
    auto full_tile = [&](lds_cptr Vp, lds_cptr Kc) {
      if (it + DIST < ntiles) issue(it + DIST);
      back(Vp);
      front(std::false_type{}, two, Kc, it * BN, 0, 0, []() {});
      wait_tile(it + 1);
      __syncthreads();
      it++;
    };
    if (NST == 4) {
      // it % NST == 1 here (or no full tile at all): copies with compile-time stages
      for (; it + NST <= n_full;) {
        full_tile(smem + BN * HD, smem + 1 * 2 * BN * HD);
        full_tile(smem + 1 * 2 * BN * HD + BN * HD, smem + 2 * 2 * BN * HD);
        full_tile(smem + 2 * 2 * BN * HD + BN * HD, smem + 3 * 2 * BN * HD);
        full_tile(smem + 3 * 2 * BN * HD + BN * HD, smem);
      }
    }
    c_st = it % NST;
    for (; it < n_full;) {
      const int prev = (c_st == 0) ? NST - 1 : c_st - 1;
      full_tile(stage_k(prev) + BN * HD, stage_k(c_st));
      c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
    }
    bool pending = it > 0;  // a tile whose V product is still to do
    int p_st = (c_st == 0) ? NST - 1 : c_st - 1;
    for (; it < ntiles; it++) {
      if (it + DIST < ntiles) issue(it + DIST);
      if (pending) back(stage_k(p_st) + BN * HD);
      pending = false;
      const bool dep = !NODEPTH && it >= n_seq;
      const int col0 = dep ? dep0 + (it - n_seq) * BN : it * BN;
      const int lo = dep ? dlo : 0;
      const int hi = dep ? dhi : shi;
      const bool touches = (hi > col0) && (lo < col0 + BN) && (hi > lo);
      if (__any(touches)) {
        front(std::true_type{}, two, stage_k(c_st), col0, lo, hi, []() {});
        pending = true;
        p_st = c_st;
      }
      c_st = (c_st + 1 == NST) ? 0 : c_st + 1;
      wait_tile(it + 1);
      __syncthreads();
    }
    if (pending) back(stage_k(p_st) + BN * HD);
  }

  if (own_depth) {
    if (!EARLY) __syncthreads();  // (EARLY: every tile ends with one)
    if (!early) enter_depth();
    const int nh = (c_end - c_beg + 31) / 32;
    // (Depth-only launches stream from memory; a second tile on its way costs them 4 %: 102 x 197 tokens of two rows, ten slots, 13.1
    // and 13.7 us.)
    if (TWO_SETS && (APART || a.has_seq)) {
      if (!early && nh > 0) fetch_early();
      for (int j = 0; j < nh; j++) {
        const int col0 = c_beg + 32 * j;
        lds_ptr Kt = own_tile(j & 1), Vt = own_v(j & 1);
        if (j + 1 < nh) {
          fetch(own_tile((j + 1) & 1), kdp, a.skd.t, col0 + 32, a.D);
          fetch(own_v((j + 1) & 1), vdp, a.svd.t, col0 + 32, a.Dv);
          next_columns();
          Own::template wait_but<3 * Own::N>();  // K landed, V may still be on its way
        } else {
          Own::template wait_but<Own::N>();
        }
        half_tile(Kt, Vt, col0, dlo, dhi, [&]() {
          if (j + 1 < nh)
            Own::template wait_but<2 * Own::N>();
          else
            Own::template wait_but<0>();
        });
        Own::reads_done();
      }
    } else if (nh > 0) {
      // The next K tile is fetched as soon as the scores are out, the next V tile once the V product is.
      lds_ptr Kt = own_tile(0), Vt = EARLY && !TWO_SETS ? own_tile(1) : Kt + 32 * HD;
      if (!early) fetch(Kt, kdp, a.skd.t, c_beg, a.D);
      fetch(Vt, vdp, a.svd.t, c_beg, a.Dv);
      for (int j = 0; j < nh; j++) {
        const int col0 = c_beg + 32 * j;
        const bool more = j + 1 < nh;
        Own::template wait_but<Own::N>();  // K landed, V may still be on its way
        front(std::true_type{}, one, Kt, col0, dlo, dhi, []() {});
        Own::reads_done();
        next_columns();
        if (more) fetch(Kt, kdp, a.skd.t, col0 + 32, a.D);
        if (more)
          Own::template wait_but<Own::N>();  // V landed, the next K on its way
        else
          Own::template wait_but<0>();
        TrPipe<T, HD, 2, 2> pv1;
        const i32x4 P1[2] = {P[0], P[1]};
        pv1.prefetch(oa, Vt);
        pv1.run(oa, Vt, P1, o);
        Own::reads_done();
        if (more) fetch(Vt, vdp, a.svd.t, col0 + 32, a.Dv);
      }
    }
  }

#ifdef MODA_SIDE_BY_SIDE
  __syncthreads();
  if (idle) return;
  // (A row past the end comes with what the unmasked tiles gave its zero query, the mean of their V rows: whoever takes the rows keeps
  // them apart and does not store it.)
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int i4 = 0; i4 < 4; i4++) {
      i32x2 w;
      w[0] = pack2<T>(o[d][4 * i4 + 0] * inv, o[d][4 * i4 + 1] * inv);
      w[1] = pack2<T>(o[d][4 * i4 + 2] * inv, o[d][4 * i4 + 3] * inv);
      out(wave * 32 + n, 4 * d + i4, g, w);
    }
#else
  if (valid) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* op = a.out_o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        i32x2 w;
        w[0] = pack2<T>(o[d][4 * i4 + 0] * inv, o[d][4 * i4 + 1] * inv);
        w[1] = pack2<T>(o[d][4 * i4 + 2] * inv, o[d][4 * i4 + 3] * inv);
        if (32 * d + 8 * i4 + 4 * g < a.Dv) *reinterpret_cast<i32x2*>(op + 32 * d + 8 * i4 + 4 * g) = w;
      }
    if (g == 0) a.lse[((int64_t)b * a.Tq + r) * a.Hq + hq] = (l > 0.f) ? m + log2f(l) : kNegInf;
  }
#endif
}

}  // namespace moda
