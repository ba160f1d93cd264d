// Compile-time launch shapes of the streaming (query-row) kernels: forward and dQ; rules of the dense ones.
#pragma once

namespace moda {

// Waves per workgroup (16 * NB query rows each; NB matters to the 16x16x32 kernels only), LDS ring stages of one 64-column K tile + V tile, and how
// many tiles ahead the global->LDS loads run.
//
// 128-wide tiles: RowLarge is the throughput shape, 256 query rows share every K/V tile, one workgroup per compute unit.
// RowSmall<128> is for problems with few query rows per (batch, head), where the large shape leaves compute units
// without a workgroup and makes every wave sit through the barriers of depth tiles that only other waves of its
// workgroup touch.
//
// 64-wide tiles: four waves (128 rows) with two ring stages of 16 KB are the better shape at every size.  Two
// workgroups of the dQ kernel and three of the forward kernel (whose registers then fit three waves per SIMD) share a
// compute unit and cover each other's softmax, depth phase, start and end, where the eight-wave workgroup of
// the 128-wide tiles is alone: forward 2.87 -> 2.47 ms and dQ 3.71 -> 3.57 ms at 16 K tokens, 64 query heads, 64 slots;
// 181 -> 145 us and 217 -> 187 us at 3 x 4 144 tokens, 16 query heads without a depth stream.
struct RowLarge {
  static constexpr int W = 8, NST = 3, DIST = 2, NB = 2;
  static constexpr bool PP = false, APART = false;
};
// RowLarge with the upper half of the workgroup running half a tile behind the lower half (see the
// forward kernel); one more ring stage keeps the previous tile's V alive for it.
struct RowLargePP {
  static constexpr int W = 8, NST = 4, DIST = 2, NB = 2;
  static constexpr bool PP = true, APART = false;
};
template <int HD>
struct RowSmall {
  static constexpr int W = 4, NST = 2, DIST = 1, NB = 2;  // 64 KB of LDS at 128, 32 KB at 64
  static constexpr bool PP = false, APART = false;
};
// 64-wide tiles, short sequences: two waves, for a row count whose last 128-row tile would be half empty.
struct RowShort {
  static constexpr int W = 2, NST = 2, DIST = 1, NB = 2;
  static constexpr bool PP = false, APART = false;
};
// ... and with a third ring stage, for dQ launches of equal, HBM-bound workgroups (see pick_short_rows).
struct RowShort3 {
  static constexpr int W = 2, NST = 3, DIST = 2, NB = 2;
  static constexpr bool PP = false, APART = false;
};

// The attention of a block with its dense part in one launch (attend_tail_kernel): the eight waves of a workgroup, or four for each of
// two key/value heads with half the ring, load the tiles; WORK of them take 32 query rows each, those of the workgroup's 64 or 32
// tokens of all the head's query heads.  Each of those has a private K and V tile apart from the ring.
template <int KV_HEADS, int WORK>
struct RowBlock {
  static constexpr int W = 8 / KV_HEADS, NST = 4 / KV_HEADS, DIST = NST - 1, NB = 2, WORKING = WORK;
  static constexpr bool PP = false, APART = true;
  static_assert(WORK >= 1 && WORK <= W, "the query rows of the workgroup's tokens over its waves");
};
// Elements of the LDS that the ring of a block's attention and then the hidden activations have (see attend_tail_kernel)
template <typename Shape, int BM>
constexpr int attend_ring() {
  constexpr int rings = 8 / Shape::W * Shape::NST * 2 * 64 * 64;
  return rings > BM * 2 * 256 ? rings : BM * 2 * 256;
}

// Head dims above 128 (tile width 256, 16x16x32 kernels only): 16 query rows per wave, so that the wave's Q (and
// dO) operands and its 256-wide accumulator still fit the register file; two ring stages of 64 KB.
struct RowWide {
  static constexpr int W = 8, NST = 2, DIST = 1, NB = 1;
  static constexpr bool PP = false, APART = false;
};

// Host side, 128-wide tiles: the small shape is used when the large one would not even give every compute unit
// two workgroups.
inline bool use_small_rows(long long rows_per_head, long long heads, int compute_units) {
  const long long large_blocks = (rows_per_head + 32 * RowLarge::W - 1) / (32 * RowLarge::W) * heads;
  return large_blocks < 2ll * compute_units;
}

// Host side, 64-wide tiles: which two-wave shape a launch takes instead of the four-wave one.
enum class ShortRows { kNone, kTwoStages, kThreeStages };
// RowShort: an odd number of 64-row tiles per head, few enough for the half-empty 128-row tile to count (at 16 tiles
// it is 3 % of the rows), and more 128-row workgroups than compute units (fewer run side by side anyway).
// 64 x 197 tokens, four query rows each, six slots: dQ 24.3 -> 22.7 us; 101 x 257, two heads of two: 92 -> 90 us.
// RowShort3: equal workgroups (not causal) in few rounds finish with a nearly empty last round unless their count fits.
// Three ring stages allow three workgroups per compute unit instead of four: taken when that wastes fewer places.
// 64 x 197 tokens, six heads, twelve slots (1536 workgroups: two rounds of 768, one and a half of 1024): dQ 127 -> 119 us.
inline ShortRows pick_short_rows(long long rows_per_head, long long heads, bool causal, int compute_units) {
  const long long tiles = (rows_per_head + 63) / 64, n = tiles * heads;
  const long long three = 3ll * compute_units, four = 4ll * compute_units;
  const auto places = [n](long long slots) { return (n + slots - 1) / slots * slots; };
  if (!causal && n > four && places(four) <= 3 * four && places(three) < places(four)) return ShortRows::kThreeStages;
  if (tiles % 2 == 1 && tiles <= 16 && (tiles + 1) / 2 * heads > compute_units) return ShortRows::kTwoStages;
  return ShortRows::kNone;
}

// Host side, linear layers: rows x features of the workgroup's tile.  Measured at 1 900 .. 12 608 rows, K 128 .. 3 072.  A
// 128 x 128 tile where its grid is one full round of two workgroups per compute unit (12 608 x 512 -> 512: 17 us, others
// 18 - 24); 128 x 64 where that still gives two each (256 -> 384: 8.7 us), with a third stage in flight for a long k loop
// in one round (1024 -> 256: 14.6 against 15.9 us); else small tiles, five workgroups per compute unit.
enum class LinearTile { k64x64, k128x64, k128x64ThreeStages, k128x128 };
inline LinearTile pick_linear_tile(long long rows, long long K, const int* features, int parts, int compute_units) {
  const auto tiles = [=](int bm, int bn) {
    long long t = 0;
    for (int i = 0; i < parts; i++) t += (features[i] + bn - 1) / bn;
    return t * ((rows + bm - 1) / bm);
  };
  const long long large = tiles(128, 128), tall = tiles(128, 64), cus = compute_units;
  if (large >= cus + cus / 4 && large <= 2 * cus) return LinearTile::k128x128;
  if (tall >= 2 * cus) return LinearTile::k128x64;
  if (tall > cus && K >= 512) return LinearTile::k128x64ThreeStages;
  return LinearTile::k64x64;
}

// Host side, a transformer block's dense part as one launch (block_tail_kernel) or as its pieces (linear and layer-norm
// launches): rows of a workgroup of the one launch ...
inline int block_tail_rows(long long rows, int compute_units) { return rows <= 32ll * compute_units ? 32 : 64; }
// ... and whether it is the faster way.  Measured as the time of stacks of four blocks, both ways in turn, at widths 128, 256, 384
// and 512, MLPs of 1, 4, 16 and 64 times the width, 200 to 25 216 rows, both types: of 312 such stacks the rule takes the faster way or
// one within 3 % of it for 286.  The others: MLPs of 16 times the width and more near the line, 3 - 14 % behind; widths 384 and 512
// with two fifths of the last round full (22 852 rows), 4 - 15 % behind at an MLP of four times the width, up to 46 % at sixteen.
// A workgroup takes its rows through all of the block's weights, which one compute unit takes in at 64 bytes a cycle, however
// few the rows are.  The pieces spread the weights over the compute units, but are seven launches, and their time grows with
// the rows.  While 32 rows each are one round, the one launch costs, in us a block and against the pieces, 16 for a million
// weights; it saves 9 of launches, 3 for 256 features of width, the hidden activations' way through memory (less in fp16, whose
// GELU is the longer one), and for 1000 rows 1 and 2.2 for a million weights.  Width 256, MLP of 1024, 200 rows: 34 us a block,
// pieces 42; MLP of 16 384: 219 and 156, at 4 632 rows 211 and 255.  Width 512, MLP of 2048, 200 rows: 78 and 56, 8 128 rows: 92
// and 112.
// With 64 rows a round that is mostly empty costs as much as a full one.  Up to width 256 that is still less than the pieces
// (16 464 rows, two workgroups more than a round: 80 and 97); 384 has to fill half of it (16 464 rows: 165 and 154, 25 216: 179
// and 217), and so has 512 in bf16 (18 912: 259 and 237, 25 216: 280 and 320).  512 in fp16 spills most registers: three
// quarters (9 259 rows: 150 and 135, 12 608: 162 and 172).
inline bool block_tail_pays(bool fp16, long long rows, long long width, long long hidden, long long kv_width, int compute_units) {
  if (block_tail_rows(rows, compute_units) == 32) {
    const double weights = 2e-6 * (double)width * (double)(width + kv_width + hidden), k = 0.256 * (double)rows / compute_units;
    return weights * (16 - 2.2 * k) < 9 + 3 * (width / 256.) + k + (fp16 ? 0.8 : 2.7) * (hidden / 1000.);
  }
  const long long last = ((rows + 63) / 64 - 1) % compute_units + 1;  // workgroups of the last round
  return width <= 256 || 4 * last >= (width > 384 && fp16 ? 3 : 2) * compute_units;
}

// Whether 32-bit byte offsets reach all of a (batch, head) slice: `rows` rows, `stride` 16-bit elements apart.
inline bool narrow_slice(long long rows, long long stride) { return 2 * rows * stride <= 0x7fffffffll; }

// ... and whether the block's attention joins it (attend_tail_kernel): workgroups of 64 (or 32) tokens of one sequence, which a
// sequence's last one has few of, as long as they take no more rounds than workgroups of as many rows of all.
// `slots`: of a token in the depth cache, whose rows are a layer's k and v as well as its depth rows.  Slices that 32-bit offsets do
// not reach are the forward kernel's alone.
// The joined launch saves a block 3.5 us of starts and ends (causal: 4.5, and 7 where 32 tokens a workgroup leave the light ones time to
// take in weights), and the attention takes as long or longer in it, which grows with the sequence.  Of 64 keys, a SIMD takes 0.73 us for
// one wave's 32 rows, 1.16 for those of two waves, 1.62 of three.  The joined launch has one workgroup a compute unit, so one
// working wave a SIMD, or two (four query heads and 64 tokens; two key/value heads, whose halves' working waves share SIMDs), round
// after round; the forward launch up to three.  Causal, a round of the one lasts as long as its longest row, while the other's
// workgroups, all there at once, make room for each other.  Over several rounds less is saved: the dense launch by itself overlaps a
// round's end with the next one's start (width 128 most of all).
// Measured: stacks of two, six and twelve blocks, both ways in turn, 20 - 65 536 tokens, one to eight rounds, causal and not, both types,
// MLPs of two to eight times the width, the heads that the kernel takes.  The rule was fitted to 1595 of them that take as many rounds
// either way; 1585 go the faster way or one within 3 % of it, and 1381 of 1398 random ones drawn afterwards, the others within 7 %, one
// 11 % behind.  Of the 1595, always joined, 373 would lose more than 3 %, up to 31 %, and always apart 805, up to 30 %.  us of six
// blocks apart and joined, one key/value head: four query heads, 64 x 197 tokens 281 and 256; causal, 1 x 16 384 1475 and 1854, 2 x 8192
// 869 and 1042, 2 x 4096 478 and 429; two query heads, 4 x 16 384 3836 and 4950, 1 x 16 384 1284 and 1256; two key/value heads of two,
// 1 x 4096 472 and 590, 4 x 4096 716 and 703.
inline bool attend_tail_takes(long long width, long long heads, long long kv_heads, long long tokens) {
  const long long group = kv_heads > 0 ? heads / kv_heads : 0;
  return (kv_heads == 1 || kv_heads == 2) && heads == group * kv_heads && (group == 2 || group == 4) && width == 64 * heads &&
         tokens * heads <= 256;  // query rows, 32 a wave
}
inline bool attention_joins_tail(long long batch, long long tokens, long long width, long long heads, long long kv_heads, long long slots,
                                 bool causal, int compute_units) {
  const long long rows = batch * tokens, bm = block_tail_rows(rows, compute_units), cus = compute_units;
  const long long tiles = (rows + bm - 1) / bm, with = batch * ((tokens + bm - 1) / bm), rounds = (with + cus - 1) / cus;
  if (!attend_tail_takes(width, heads, kv_heads, bm) || !narrow_slice(tokens, slots * kv_heads * 64) || rounds != (tiles + cus - 1) / cus) return false;
  constexpr double one = 0.73, two = 1.16, three = 1.62;
  const double keys = (double)((tokens + 63) / 64);  // tiles of the longest row
  const bool pairs = kv_heads == 2 || bm * heads > 128;  // waves at work two a SIMD
  const double joined = (pairs ? two : one) * (!causal ? (double)rounds : with > 2 * cus ? 0.5 * with / cus : 1);
  // the forward launch's workgroups, 128 rows each, a compute unit; up to three are there at once
  const double n = (double)(batch * kv_heads * ((tokens * (heads / kv_heads) + 127) / 128)) / cus;
  double apart;
  if (n > 3) {
    apart = three / 3 * n * (causal ? 0.5 : 1);
  } else if (causal) {  // those of the unit that has the longest row: the second and third have so much of it
    const double second = n > 1 ? 1 - 1 / n : 0, third = n > 2 ? 1 - 2 / n : 0;
    apart = third * three + (second - third) * two + (1 - second) * one;
  } else {
    apart = n <= 1 ? one : n <= 2 ? two : three;
  }
  if (rounds > 2 && !pairs) return false;
  const double saved = rounds == 1 ? (!causal ? 3.5 : bm == 32 ? 7 : 4.5) : !pairs ? 1.3 : causal ? 4 : kv_heads == 1 ? 3.5 : 2;
  return (joined - apart) * keys <= saved + 1e-6;
}

}  // namespace moda
