// Index arithmetic of the attention kernels: which rows and columns a workgroup, a wave and a lane touch.
// Everything here is plain integer code marked for host and device, shared by the kernels, their host
// launchers and the host-side address walker of the test suite (tests/address_walker.cpp), which replays
// every descriptor, load and store of a launch on the CPU and checks them against the tensor extents.
#pragma once
#include "kargs.h"
#include "tuning.h"

#define MODA_HD __host__ __device__ __forceinline__

namespace moda {

MODA_HD int imin(int a, int b) { return a < b ? a : b; }
MODA_HD int imax(int a, int b) { return a > b ? a : b; }

// Depth columns.  A depth tensor holds L slots per token (row t * L + l = slot l of token t) of which the first
// Lv hold data.  The kernels count depth columns on the COMPACT axis of the slots that hold data: column
// c = t * Lv + l; slots l >= Lv are never read.  With Lv == L (every slot filled) the compact axis is the row axis.
MODA_HD int64_t depth_row_of(const KArgs& a, int c) {
  if (a.Lv == a.L) return c;
  const int t = c / a.Lv;
  return (int64_t)t * a.L + (c - t * a.Lv);
}

// ---------------------------------------------------------------------------------------------------
// Query-row kernels (forward, dQ): a workgroup owns BM consecutive query rows of one (batch, query head)
// and streams BN-column tiles: the sequence keys, then (when they go through the workgroup's ring) the
// depth columns its rows can see.
// ---------------------------------------------------------------------------------------------------

// Query tile of workgroup `block` (heavy, late tiles first).  In a variable-length batch the grid counts tiles
// from the end of the longest sequence (Tq_longest), so that tiles of equal cost of all sequences are dispatched
// together; a result >= the sequence's own tile count means the workgroup has nothing to do.
MODA_HD int query_tile_of(int block, int BH, int BM, int Tq_grid) { return (Tq_grid + BM - 1) / BM - 1 - block / BH; }

// Packed order: the tiles of all sequences of a packed batch as one list, by cost level (row kernels: the tile's index;
// dK/dV: how many column tiles lie behind it), the highest level first and the sequences that reach a level in turn; the
// heads of a tile are neighbours in the grid.  (Cost in a causal batch; where every row sees all keys a tile costs what its
// sequence is long, and the levels only mix the sequences.)  A workgroup finds its place itself: N(j) = sum of max(0, tiles - j) counts
// the list's entries at level j or above, its level is the largest j with N(j) > rank.
// What it replaces, a grid of the longest sequence for every one, launched mostly workgroups without work on unequal
// lengths, and sent a (sequence, head) to the XCD that its index fell on (block % 8): with B * H a multiple of 8 the longest
// sequence's tiles stayed on as many XCDs as it has heads.  Training steps: 16 sequences of 113 - 7441 tokens, two heads of
// four, head dim 64: 3480 -> 737 us; twelve of 338 - 7523, four heads of two: 1296 -> 666; 8192 + 3 x 64 tokens, two heads of
// two, head dim 128: 1139 -> 766; 16 384 to 2048 tokens, 15 sequences, four heads of four: 10.14 -> 9.84 ms; 200 of 300 each:
// 1710 -> 1671 us.
// Two kinds of launches keep that grid.  Those of up to kPackedOrderGrid workgroups in it, where every workgroup has a compute
// unit to itself wherever it falls: a place in the list costs a launch 0.4 us (forward of 8 x 14 - 262 tokens, four heads of
// two, head dim 64: 9.4 us in the list, 9.0 in the grid; two of up to 147, eight heads of four: 8.2 and 7.8).  Above, the list's
// order is worth more than that (5909 + 433 tokens, four heads, a grid of 376: 108 -> 78).  And those of more than
// kPackedOrderMax sequences, whose tile counts a wave holds in four registers (one up to 64: 0.3 us less).
// What is left of the list's price: launches whose workgroups all run at once, two or three a compute unit, end by which of
// them share one (226, 1800, 6188, 900, 3300 tokens, two heads of two, head dim 64, causal: 268 -> 271 us a step, not causal with
// four slots 426 -> 413; 12 of 1332 and fewer, four heads: 91 -> 93).
constexpr int kPackedOrderMax = 256, kPackedOrderGrid = 256;
// workgroups of the grid of the longest sequence for every one
MODA_HD int64_t longest_row_grid(const KArgs& a, int BM) { return (int64_t)((a.Tq + BM - 1) / BM) * a.B * a.Hq; }
MODA_HD int64_t longest_col_grid(const KArgs& a, int BN, int nseg) { return a.has_seq ? (int64_t)((a.T + BN - 1) / BN) * nseg * a.B * a.Hkv : 0; }
MODA_HD bool packed_order(const KArgs& a, int64_t grid) { return a.cu != nullptr && a.B <= kPackedOrderMax && grid > kPackedOrderGrid; }
// length of the list, at most: every sequence has one tile that is not full (rows_per_token: query rows, or 1 for keys)
MODA_HD int64_t packed_ranks(const KArgs& a, int rows_per_token, int BM) {
  const int64_t grid = (int64_t)(((int64_t)a.T * rows_per_token + BM - 1) / BM) * a.B;
  const int64_t list = (int64_t)(a.delta_pitch / a.Gf) * rows_per_token / BM + a.B;
  return grid < list ? grid : list;
}
struct PackedTile {
  int seq, level;
  int t0, T;    // the sequence's first token and length
  bool active;  // false: past the end of the list
};
template <int P>  // sequences: up to 64 P
MODA_HD PackedTile packed_tile_of(const KArgs& a, int rows_per_token, int BM, int rank) {
  PackedTile p = {0, 0, 0, 0, false};
#if defined(__HIP_DEVICE_COMPILE__)
  const int lane = threadIdx.x & 63;
  int tiles[P], t0[P], T[P];
#pragma unroll
  for (int i = 0; i < P; i++) {
    const int s = 64 * i + lane;
    t0[i] = T[i] = 0;
    if (s < a.B) {
      t0[i] = a.cu[s];
      T[i] = a.cu[s + 1] - t0[i];
    }
    tiles[i] = (T[i] * rows_per_token + BM - 1) / BM;
  }
  const auto entries_from = [&](int j) {  // N(j)
    int x = 0;
#pragma unroll
    for (int i = 0; i < P; i++) x += imax(0, tiles[i] - j);
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8: sums of 16 lanes
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast 15, 31: lane 63 holds all
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return __builtin_amdgcn_readlane(x, 63);
  };
#else
  const auto tiles_of = [&](int s) { return ((a.cu[s + 1] - a.cu[s]) * rows_per_token + BM - 1) / BM; };
  const auto entries_from = [&](int j) {
    int x = 0;
    for (int s = 0; s < a.B; s++) x += imax(0, tiles_of(s) - j);
    return x;
  };
#endif
  if (entries_from(0) <= rank) return p;
  int lo = 0, hi = (a.T * rows_per_token + BM - 1) / BM, above = 0;  // N(lo) > rank >= N(hi) = above
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2, n = entries_from(mid);
    if (n > rank) {
      lo = mid;
    } else {
      hi = mid;
      above = n;
    }
  }
  p.level = lo;
  int nth = rank - above;  // among the sequences that reach the level
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < P; i++) {
    const uint64_t there = __builtin_amdgcn_ballot_w64(tiles[i] > lo);
    const int count = __builtin_popcountll(there);
    if (!p.active && nth < count) {
      const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(there >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)there, 0));
      const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(tiles[i] > lo && before == nth));
      p.seq = 64 * i + at;
      p.t0 = __builtin_amdgcn_readlane(t0[i], at);
      p.T = __builtin_amdgcn_readlane(T[i], at);
      p.active = true;
    }
    nth -= count;
  }
#else
  for (int s = 0; s < a.B && !p.active; s++)
    if (tiles_of(s) > lo && nth-- == 0) {
      p.seq = s;
      p.t0 = a.cu[s];
      p.T = a.cu[s + 1] - p.t0;
      p.active = true;
    }
#endif
  return p;
}
MODA_HD PackedTile packed_tile(const KArgs& a, int rows_per_token, int BM, int rank) {
  return a.B <= 64 ? packed_tile_of<1>(a, rows_per_token, BM, rank) : packed_tile_of<kPackedOrderMax / 64>(a, rows_per_token, BM, rank);
}

// Which (batch entry, query head, query tile) a workgroup of the forward or dQ kernel takes.
struct RowPlace {
  int b, hq, qt;
  int t0, T;  // packed batch: the sequence's first token and length
  bool active;
};
template <bool VARLEN>
MODA_HD RowPlace row_place(const KArgs& grid, int block, int BM) {
  if (VARLEN && packed_order(grid, longest_row_grid(grid, BM))) {
    const PackedTile p = packed_tile(grid, grid.Gf, BM, block / grid.Hq);
    return {p.seq, block % grid.Hq, p.level, p.t0, p.T, p.active};
  }
  const int BH = grid.B * grid.Hq, bh = block % BH;
  const int b = bh / grid.Hq, qt = query_tile_of(block, BH, BM, grid.Tq);
  const int t0 = VARLEN ? grid.cu[b] : 0, T = VARLEN ? grid.cu[b + 1] - t0 : grid.T;
  return {b, bh % grid.Hq, qt, t0, T, !VARLEN || qt < (T * grid.Gf + BM - 1) / BM};
}

// Which tokens a workgroup of attend_tail_kernel takes: tile `tile` (of `tokens` each) of sequence b, rows [first_row, rows_end) of
// the [B * T] rows; a sequence's tiles are B workgroups apart, on one XCD (one L2) if B is a multiple of eight.  Causal: the late, heavy
// tiles first, as in query_tile_of.  Six blocks of width 256 on causal sequences, us with the light ones first and so: 4 x 8192 tokens
// (two rounds) 1654 and 1360, 1 x 65 536 (four) 20 440 and 15 290, 64 x 512 (two) 517 and 505; one round 1864 and 1854 (1 x 16 384).
struct AttendTailPlace {
  int b, tile, first_row, rows_end;
};
MODA_HD AttendTailPlace attend_tail_place(const KArgs& a, int block, int tokens) {
  const int nth = block / a.B, b = block % a.B, tile = a.causal ? (a.T + tokens - 1) / tokens - 1 - nth : nth;
  return {b, tile, b * a.T + tile * tokens, (b + 1) * a.T};
}
inline int64_t attend_tail_blocks(const KArgs& a, int tokens) { return (int64_t)a.B * ((a.T + tokens - 1) / tokens); }

// Workgroups of the launch that packs weights (`packing` for each of `parts`) and normalises rows (pack_and_norm_kernel), or 0 where the
// 2^32 threads of a grid's one dimension do not hold both: two launches then, as large as each may be by itself.
inline int64_t pack_and_norm_blocks(int64_t rows, int rows_per_block, int64_t packing, int64_t parts) {
  const int64_t n = (rows + rows_per_block - 1) / rows_per_block + packing * parts;
  return n * 256 < (1ll << 32) ? n : 0;
}

// Visible column intervals [0, shi) of the sequence keys and [dlo, dhi) of the depth columns (compact axis) for
// query row r (all zero for a row past the end).  Ld: depth slots per token, 0 when the launch has no depth stream.
struct RowVis {
  int shi, dlo, dhi;
};
MODA_HD RowVis row_visibility(const KArgs& a, int r, int Ld) {
  RowVis v = {0, 0, 0};
  if (r < a.Tq) {
    const int t = r / a.Gf;
    if (a.has_seq) v.shi = a.causal ? t + 1 : a.T;
    if (Ld > 0) {
      const int lo_t = a.chunk ? (t / a.Cb) * a.Cb : t;
      v.dlo = lo_t * a.Lv;
      v.dhi = (t + 1) * a.Lv;
    }
  }
  return v;
}

// Depth columns a wave alone can see (always outside chunk-visible mode, and in it when a chunk's rows fit a
// wave pair) are not streamed through the workgroup's ring: each wave fetches its own rows' span.
MODA_HD bool waves_own_depth(const KArgs& a, int Ld) { return Ld > 0 && (!a.chunk || a.Cb * a.Gf <= 64); }

// Outside chunk-visible mode a depth slot is seen by the Gf query rows of its own token only.  When those rows
// always sit in one wave of the dQ kernel (32 rows per wave, Gf divides 32) the dQ kernel can form the slots' dK
// and dV while their K and V rows are in its LDS tiles: no other wave contributes to them, and the depth stream is
// read once per backward instead of twice.  Done for the 64-wide tiles only -- there the extra operands (Q^T and
// dO^T of the wave's rows) fit the register file next to the dQ accumulators, and the shapes that use them are
// bound by memory traffic; on the 128-wide tiles the same code spills and was measured slower than the separate
// depth-column kernel, which every other case runs from the dK/dV launch.
constexpr int kDepthGradsInDqMaxWidth = 64;
MODA_HD bool depth_grads_in_dq(const KArgs& a, int HD) {
  return a.L > 0 && !a.chunk && HD <= kDepthGradsInDqMaxWidth && 32 % a.Gf == 0 && !a.far_depth_grads;
}

// ... and where the dQ kernel's waves walk their own depth columns without forming the gradients (the 128-wide tiles,
// or a query group that does not divide a wave), they can at least hand their rounded P and dS of the (row, slot)
// pairs to the depth-column kernel through the workspace (KArgs::depth_p), which then skips reading kd, vd and
// recomputing the scores.
MODA_HD bool depth_scores_from_dq(const KArgs& a, int HD) {
  return a.L > 0 && !a.chunk && HD <= 128 && !depth_grads_in_dq(a, HD);
}

// Private depth tiles that are sent for while the last ring tile, in stage `last`, is worked on: the first of two sets, or of K and V
// places, that lies outside of that stage.  Forward: a set is one of two stages.  dQ with the depth gradients: a set is a stage of two
// or three, or (four waves) as large as the whole ring.
MODA_HD int fwd_first_private_set(int last) { return last ^ 1; }
MODA_HD int dq_first_private_set(int waves, int last) { return waves > 2 || last == 0 ? 1 : 0; }

// The column tiles of query tile qt: n_seq sequence tiles, of which the first n_full are seen completely by every
// row of the workgroup, then n_dep depth tiles starting at flattened depth column dep0 (ring_depth: the depth
// columns go through the ring at all).
struct RowTilePlan {
  int n_seq, n_full, dep0, n_dep;
};
MODA_HD RowTilePlan row_tile_plan(const KArgs& a, int qt, int BM, int BN, bool ring_depth) {
  RowTilePlan p = {0, 0, 0, 0};
  const int r_first = qt * BM;
  const int r_last = imin(a.Tq, r_first + BM) - 1;
  const int t_first = r_first / a.Gf, t_last = r_last / a.Gf;
  if (a.has_seq) {
    p.n_seq = ((a.causal ? t_last + 1 : a.T) + BN - 1) / BN;
    // padding rows of the last workgroup compute on zero queries in the full tiles and are never stored
    p.n_full = imin(p.n_seq, (a.causal ? t_first + 1 : a.T) / BN);
  }
  if (ring_depth) {
    const int lo_t = a.chunk ? (t_first / a.Cb) * a.Cb : t_first;
    p.dep0 = lo_t * a.Lv;
    p.n_dep = ((t_last + 1) * a.Lv - p.dep0 + BN - 1) / BN;
  }
  return p;
}
// first row (sequence key or flattened depth column) of ring tile `it`
MODA_HD int ring_tile_row0(const RowTilePlan& p, int it, int BN) {
  return it < p.n_seq ? it * BN : p.dep0 + (it - p.n_seq) * BN;
}

// Depth columns [c_beg, c_end) that the `rows` query rows starting at rw0 (< Tq) can see.
struct DepthSpan {
  int c_beg, c_end;
  int t_beg;  // token of the first one
};
MODA_HD DepthSpan own_depth_span(const KArgs& a, int rw0, int rows) {
  const int tw0 = rw0 / a.Gf, tw1 = (imin(a.Tq, rw0 + rows) - 1) / a.Gf;
  DepthSpan s;
  s.t_beg = a.chunk ? (tw0 / a.Cb) * a.Cb : tw0;
  s.c_beg = s.t_beg * a.Lv;
  s.c_end = (tw1 + 1) * a.Lv;
  return s;
}

// ---------------------------------------------------------------------------------------------------
// Column kernel (dK/dV): a workgroup owns BN columns -- sequence keys or flattened depth columns -- of one
// (batch, kv head) and streams BM-row query tiles from the last visible one down.
// ---------------------------------------------------------------------------------------------------

// visible query-row interval [lo, hi) of a column
MODA_HD void q_interval(const KArgs& a, bool dep, int col, int& lo, int& hi) {
  if (!dep) {
    lo = a.causal ? col * a.Gf : 0;
    hi = a.Tq;
  } else {
    const int w = col / a.Lv;
    lo = w * a.Gf;
    hi = a.chunk ? imin(a.T, (w / a.Cb + 1) * a.Cb) * a.Gf : (w + 1) * a.Gf;
  }
}

// What column-tile workgroup `ct` of a (batch, kv head) does.  `grid`: the launch's argument block (T of the
// longest sequence), `a`: the one rebased on the workgroup's sequence; nseg: row segments per sequence tile.
struct ColTilePlan {
  bool active;  // false: a tile beyond this sequence of a variable-length batch, or a segment a tile does without
  bool dep;     // depth columns (else sequence keys)
  int ncols;    // columns of the (batch, head): T or T * L
  int seg;      // row segment of a split sequence tile ...
  int nsegs;    // ... out of this many (1: the workgroup writes the gradients itself)
  int c_first;  // first column
  int qt0, nqt; // query tiles qt0 .. qt0 + nqt - 1 (BM rows each), streamed from the last one down
};
// row segments of a sequence column tile that sees `nqt` query tiles
MODA_HD int tile_segments(const KArgs& grid, int nqt, int nseg) {
  return grid.dkv_seg_tiles > 0 ? imax(1, imin(nseg, (nqt + grid.dkv_seg_tiles - 1) / grid.dkv_seg_tiles)) : nseg;
}
MODA_HD ColTilePlan col_tile_plan(const KArgs& grid, const KArgs& a, int ct, int BN, int BM, bool varlen, int nseg) {
  ColTilePlan p;
  // the grid holds the sequence tiles of the longest sequence (nseg workgroups each: the row segments of one
  // column tile are neighbours in the grid), then, when launched with them, the depth tiles
  const int n_seq_tiles = grid.has_seq ? (grid.T + BN - 1) / BN : 0;
  p.active = true;
  p.dep = ct >= n_seq_tiles * nseg;
  p.ncols = p.dep ? a.T * a.Lv : a.T;
  p.seg = p.dep ? 0 : ct % nseg;
  int tile = p.dep ? ct - n_seq_tiles * nseg : ct / nseg;
  if (varlen && !p.dep && a.causal) {
    // a causal sequence tile costs what lies behind it: count the grid's tiles from the end of the sequence, so
    // that tiles of equal cost of all sequences are dispatched together, the heaviest of the whole batch first
    tile -= n_seq_tiles - (a.T + BN - 1) / BN;
    if (tile < 0) p.active = false;
  }
  p.c_first = tile * BN;
  if (varlen && p.c_first >= p.ncols) p.active = false;
  p.qt0 = p.nqt = 0;
  p.nsegs = 1;
  if (!p.active) return p;
  int wg_lo, wg_hi, tmp;
  q_interval(a, p.dep, p.c_first, wg_lo, tmp);
  q_interval(a, p.dep, imin(p.ncols, p.c_first + BN) - 1, tmp, wg_hi);
  p.qt0 = wg_lo / BM;
  p.nqt = (wg_hi + BM - 1) / BM - p.qt0;
  if (nseg > 1 && !p.dep) {  // this workgroup's share of the column tile's query tiles
    p.nsegs = tile_segments(grid, p.nqt, nseg);
    if (p.seg >= p.nsegs) p.active = false;
    const int lo = (int)((int64_t)p.nqt * p.seg / p.nsegs), hi = (int)((int64_t)p.nqt * (p.seg + 1) / p.nsegs);
    p.qt0 += lo;
    p.nqt = hi - lo;
  }
  return p;
}

// Which (batch entry, kv head, column-tile workgroup `ct` of it) a workgroup of the dK/dV kernels takes.  A batch in packed
// order has the sequence tiles of all its sequences first, then the depth tiles as every other launch has them.
// Row segments: the last one of every tile first, then the one before it, so that the long tiles, which alone have many,
// still lead, and the places of segments that a tile does without lie together.  Side by side, as the other launches have
// them, those places repeat with a period that compute units and XCDs share: the fullest XCD had 1.34 - 1.45 of the mean work
// (here 1.02).  dK/dV stage, causal, head dim 64, the longest sequence's grid / side by side / here: 2667 and two shorter
// sequences, eight heads 73 / 82 / 64 us; 3825 and two, one head of four 96 / 108 / 74; 1497 and four, two heads of four 56 / 64 / 57.
struct ColPlace {
  int b, hkv, ct;
  int t0, T;
  bool active;
};
template <bool VARLEN>
MODA_HD ColPlace col_place(const KArgs& grid, int block, int BN, int nseg) {
  const int BHk = grid.B * grid.Hkv;
  int ct0 = 0;
  if (VARLEN && packed_order(grid, longest_col_grid(grid, BN, nseg))) {
    const int n_seq_tiles = grid.has_seq ? (grid.T + BN - 1) / BN : 0;
    const int ranks = grid.has_seq ? (int)packed_ranks(grid, 1, BN) : 0, seq_blocks = ranks * nseg * grid.Hkv;
    if (block < seq_blocks) {
      const int place = block / grid.Hkv, seg = nseg - 1 - place / ranks;
      const PackedTile p = packed_tile(grid, 1, BN, place % ranks);
      const int tile = grid.causal ? n_seq_tiles - 1 - p.level : p.level;  // as col_tile_plan counts them
      return {p.seq, block % grid.Hkv, tile * nseg + seg, p.t0, p.T, p.active};
    }
    block -= seq_blocks;
    ct0 = n_seq_tiles * nseg;
  }
  const int bh = block % BHk, b = bh / grid.Hkv;
  const int t0 = VARLEN ? grid.cu[b] : 0, T = VARLEN ? grid.cu[b + 1] - t0 : grid.T;
  return {b, bh % grid.Hkv, ct0 + block / BHk, t0, T, true};
}

// rows of query tile starting at row f_q0 that exist (only a head's top tile can be short)
MODA_HD int query_tile_rows(const KArgs& a, int f_q0, int BM) { return imax(imin(a.Tq - f_q0, BM), 0); }

// ---------------------------------------------------------------------------------------------------
// Linear layers: the feature tiles of one row tile go to one XCD (blocks b, b + 8, b + 16, ... share an L2), which reads
// its input rows once.  Row tiles past the last one have nothing to do.
// ---------------------------------------------------------------------------------------------------
MODA_HD int linear_row_tile(unsigned block, int n_tiles) { return (int)(block & 7) + 8 * ((int)(block >> 3) / n_tiles); }
MODA_HD int linear_feature_tile(unsigned block, int n_tiles) { return (int)(block >> 3) % n_tiles; }
inline int64_t linear_blocks(int m_tiles, int n_tiles) { return 8ll * ((m_tiles + 7) / 8) * n_tiles; }

// ---------------------------------------------------------------------------------------------------
// Launch grids (host side), one place for the launchers and the walker.
// ---------------------------------------------------------------------------------------------------
inline int64_t row_kernel_blocks(const KArgs& a, int rows_per_block) {
  const int64_t grid = longest_row_grid(a, rows_per_block);
  return packed_order(a, grid) ? packed_ranks(a, a.Gf, rows_per_block) * a.Hq : grid;
}
// chunk-visible depth columns: by whole chunks when a chunk's rows fit one 64-row query tile (tile widths up to 128:
// the chunk kernel's registers and LDS do not stretch to 256), else as column tiles of the dK/dV kernel
inline bool depth_by_chunks(const KArgs& a, int HD) { return HD <= 128 && a.L > 0 && a.chunk && (int64_t)a.Cb * a.Gf <= 64; }
// workgroups for the sequence column tiles of a launch
inline int64_t seq_col_blocks(const KArgs& a, int BN, int nseg) {
  const int64_t grid = longest_col_grid(a, BN, nseg);
  return packed_order(a, grid) ? packed_ranks(a, 1, BN) * nseg * a.Hkv : grid;
}
inline int64_t col_kernel_blocks(const KArgs& a, int HD, int BN, int nseg) {
  const int64_t n_dep_tiles = (a.L > 0 && a.chunk && !depth_by_chunks(a, HD)) ? ((int64_t)a.T * a.Lv + BN - 1) / BN : 0;
  return seq_col_blocks(a, BN, nseg) + n_dep_tiles * a.B * a.Hkv;
}
// Sequence dK/dV on the 64-wide tiles: dkv_flat_kernel (three workgroups per compute unit, where dkv_kernel fits one)
// takes every launch of sequence-key column tiles whose kv head is the query head.
inline int64_t dkv_flat_blocks(const KArgs& a, int BN = 128, int nseg = 1) { return seq_col_blocks(a, BN, nseg); }
inline bool takes_dkv_flat(const KArgs& a, int HD) {
  return HD == 64 && a.has_seq && a.hdiv == 1 && col_kernel_blocks(a, HD, 128, 1) == dkv_flat_blocks(a);
}
// ... with the four waves on the SAME 32 columns and a quarter of every 128-row query tile each, for short launches whose
// 128-column tiles would leave compute units idle (64 x 197 tokens of four query rows: 128 tiles; the twelve layers of a
// depth stream 925 -> 810 us).  Longer ones are cut into segments, which re-read the query rows less.
constexpr int kDkvRowWavesMaxRows = 1024;
inline bool dkv_flat_row_waves(const KArgs& a) {
  return !a.cu && a.Tq <= kDkvRowWavesMaxRows && dkv_flat_blocks(a) <= 256;
}

// whether every streamed (batch, head) slice spans less than 2 GiB
inline bool narrow_slices(const KArgs& a) {
  const int64_t seq = (int64_t)a.T * (a.sk.t > a.sv.t ? a.sk.t : a.sv.t), dep = (int64_t)a.T * a.L * (a.skd.t > a.svd.t ? a.skd.t : a.svd.t);
  return narrow_slice(1, seq > dep ? seq : dep);
}
// dQ and sequence dK/dV of the 64-wide tiles in one launch (bwd_short_kernel): row waves, and the workgroups of both run at once,
// two a compute unit.  A replayed backward pass of 48 random such shapes takes 0.71 - 0.99 of the two launches' time (one of
// 16 us 1.07), 0.75 - 0.88 where the launch holds 300 - 512 workgroups.  More than that and the launch is longer than the two (64 x 197 tokens, six heads, twelve slots: step 191 ->
// 206 us; the twelve layers of a depth stream over 64 x 197 tokens of four query rows: 734 -> 794), each of which then has
// the occupancy that its own registers and LDS allow.
constexpr int kBwdShortRows = 128;  // query rows of a dQ workgroup there
inline bool bwd_one_launch(const KArgs& a, int HD) {
  return takes_dkv_flat(a, HD) && dkv_flat_row_waves(a) && a.dkv_split <= 1 && a.own_delta && narrow_slices(a) &&
         row_kernel_blocks(a, kBwdShortRows) + dkv_flat_blocks(a, 32) <= 2 * a.compute_units;
}

// fp32: whether dQ and dK/dV go as one launch: all workgroups run at once (one per compute unit; head dims above 64 have dK/dV
// workgroups of another size).  More than that and the row sums, formed twice, cost more than the launch.  Twelve random
// shapes, replayed: 0.65 - 0.91 of the two launches.
inline bool fp32_one_launch(const KArgs& a) {
  const int64_t cols = (a.has_seq ? (a.T + 15) / 16 : 0) + ((int64_t)a.T * a.Lv + 127) / 128;
  return a.D <= 64 && a.Dv <= 64 && ((int64_t)(a.Tq + 15) / 16 * a.Hq + cols * a.Hkv) * a.B <= a.compute_units;
}

// Row segments of the sequence dK/dV launch (KArgs::dkv_split, dkv_seg_tiles): a launch ends with its longest workgroup,
// and one with few column tiles leaves compute units idle.  Sized for 256 compute units whatever the partition mode, so
// that the workspace size depends on the problem alone.
// Launches with two column tiles per compute unit (dkv_flat_kernel: per workgroup place) are not cut: dispatched heaviest
// first they balance by themselves, and the partial sums only cost (16 K tokens, sixteen query heads on four: 4.07 -> 4.97
// ms; head dim 64, 64 heads: 10.4 -> 10.9 ms).  Below that:
// dkv_kernel, fixed length: the same power of two for every tile, segments of the heaviest of at least 16 trips (a trip:
// one query tile of one query head).  3057 tokens, 32 query heads on four: 538 -> 430 us when the heads count as trips.
// While compute units have no workgroup at all, of at least 4: the serial chain of the longest is all there is (training steps, 16
// and 4: 710 tokens, four heads of four, 16 slots 123 -> 101 us; 1500, two of two, eight slots 142 -> 121; 900, sixteen query
// heads on four 116 -> 87; at least 6 or 10: up to 8 % more).
// dkv_kernel, packed, tiles wider than 64: not cut.  There a packed batch returns bit for bit what separate calls return
// that have no room for segments, and that is kept although the cut is faster (a training step of 2600 + 168 + 900 + 400
// + 1500 tokens, four heads of four, eight slots: 329 us cut, 435 not; of 6000 + 3000 + 500, two heads of four: 641, 894).
// The rest (dkv_flat_kernel; packed batches on the 64-wide tiles): segments of equal length, three quarters of a place's
// share of all trips (0.35 to 1 measure within 4 %).  A packed batch counts as one of equal, longest sequences.  Eight
// sequences of 200 - 3000 tokens, head dim 64: 974 -> 705 us; 6000 tokens, four heads of four, head dim 64: 497 -> 430 us.
struct DkvSplit {
  int nseg, seg_tiles;
};
inline DkvSplit dkv_split_plan(const KArgs& a, int HD) {
  const bool flat = takes_dkv_flat(a, HD);
  if (!a.has_seq || a.T == 0 || (flat && dkv_flat_row_waves(a)) || (a.cu && HD > 64)) return {1, 0};
  const int BN = HD > 128 ? 64 : 128, BM = flat || HD > 128 ? 32 : 64;
  const int64_t tiles = (int64_t)((a.T + BN - 1) / BN) * a.Hkv * (a.cu ? imax(1, part_rows(a) / a.T) : a.B);
  const int64_t nqt = (a.Tq + BM - 1) / BM;
  if (tiles >= (flat ? 768 : 512)) return {1, 0};
  if (!flat && !a.cu) {
    int s = 1;
    while (tiles * s < 512 && s < 8 && nqt * a.hdiv / (2 * s) >= (tiles * s < 256 ? 4 : 16) && nqt >= 2 * s) s *= 2;
    return {s, 0};
  }
  const int64_t trips = tiles * (a.causal ? (nqt + 1) / 2 : nqt) * a.hdiv / (flat ? 768 : 256);  // of one place
  const int64_t least = flat ? 24 : 40;  // trips that pay for a workgroup's start, end and partial sums
  const int64_t seg = imax((int)((trips * 3 / 4 > least ? trips * 3 / 4 : least) / a.hdiv), (int)((nqt + 15) / 16));
  const int64_t n = seg > 0 ? (nqt + seg - 1) / seg : nqt;
  return n > 1 ? DkvSplit{(int)n, (int)imax(1, (int)seg)} : DkvSplit{1, 0};
}
inline int64_t delta_kernel_blocks(const KArgs& a, int rows_per_block) {
  return (int64_t)((a.Tq + rows_per_block - 1) / rows_per_block) * a.B * a.Hq;
}

}  // namespace moda
