// A block's attention and its dense part (block_tail_kernel.hip) in one launch, without gradients: a workgroup takes the query rows of
// 64 (or 32) tokens of a sequence, two or four heads of 64 on each of one or two key/value heads, through the forward kernel's body (fwd.h)
// and leaves their attention output in LDS, where the dense part takes it up.  Bits as from the two launches.  For short sequences, and long
// ones of one round: tuning.h, attention_joins_tail, says which and what they take either way.
//
// Both launches are short, and a good part of a short launch is its start and end.  Twelve blocks of width 256 on 64 x 197 tokens: 557 ->
// 516 us.  Six blocks, apart and joined: 64 x 197 tokens 281 and 256 (fp16 312 and 281), 16 x 197 206 and 184, 8 x 50 194 and 172, 2 x
// 8192 1134 and 1086; width 128, 64 x 197 178 and 153, 4 x 197 139 and 119; two key/value heads, width 256, 64 x 197 298 and 283, 36 x 197
// 239 and 217, width 512, 36 x 197 508 and 486.  Of 92 k cycles of the largest (width 256, eleven slots) 9.7 k are the first
// loads, 12.6 k four tiles of keys, 9 k three private tiles of depth slots, the rest the dense part.  What the dense part wants from memory
// at its start, the residual rows and the table, travels with the attention's first tiles and waits in registers; ring and private K tiles
// lie where the hidden activations and the rows go later.  Registers of a wave: all 256 with 64 rows of width 256 and the norm before the
// block, where bf16 spills five to seven; width 512 in fp16 eleven; no others, but 45 - 69 scalar ones with a depth stream.  Tried: no
// barriers where the ring holds all tiles, a higher priority for every second wave of a SIMD: 519 and 521 us where this takes 517.
#define MODA_SIDE_BY_SIDE
#include "block_tail.h"

namespace moda {

namespace {

template <typename T, int C, int NB, int KV_HEADS, bool POST, int ADDR>
hipError_t launch_attend_tail_t(const TailArgs& a, const KArgs& att, hipStream_t stream) {
  constexpr int BM = 16 * NB, WORK = BM * (C / 64) / 32;  // working waves of all heads
  typedef RowBlock<KV_HEADS, WORK / KV_HEADS> Shape;
  constexpr size_t smem = table_bytes<T>() + (size_t)(BM * C + attend_ring<Shape, BM>() + WORK * 32 * 64) * sizeof(uint16_t);
  static_assert(WORK * 32 * 64 <= BM * C && smem <= 160 * 1024, "a working wave's private K tile where the rows go later, its V tile behind the ring");
  static LdsAttrState attr;
  const hipError_t e = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&attend_tail_kernel<T, C, NB, POST, ADDR, KV_HEADS>), smem);
  if (e != hipSuccess) return e;
  const int64_t nblk = attend_tail_blocks(att, BM);
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((attend_tail_kernel<T, C, NB, POST, ADDR, KV_HEADS>), dim3((unsigned)nblk), dim3(512), smem, stream, a, att);
  return hipGetLastError();
}
template <typename T, int C, int NB, int KV_HEADS>
hipError_t launch_attend_tail_as(const TailArgs& a, bool post, const KArgs& att, hipStream_t stream) {
  if (att.L == 0) return post ? launch_attend_tail_t<T, C, NB, KV_HEADS, true, 4>(a, att, stream) : launch_attend_tail_t<T, C, NB, KV_HEADS, false, 4>(a, att, stream);
  return post ? launch_attend_tail_t<T, C, NB, KV_HEADS, true, 8>(a, att, stream) : launch_attend_tail_t<T, C, NB, KV_HEADS, false, 8>(a, att, stream);
}
template <typename T>
hipError_t launch_attend_tail_of(const TailArgs& a, bool post, const KArgs& att, hipStream_t stream) {
  const bool half = block_tail_rows(a.rows, att.compute_units) == 32;
  if (att.Hkv == 1 && att.Gf == 2) return half ? launch_attend_tail_as<T, 128, 2, 1>(a, post, att, stream) : launch_attend_tail_as<T, 128, 4, 1>(a, post, att, stream);
  if (att.Hkv == 1) return half ? launch_attend_tail_as<T, 256, 2, 1>(a, post, att, stream) : launch_attend_tail_as<T, 256, 4, 1>(a, post, att, stream);
  if (att.Gf == 2) return half ? launch_attend_tail_as<T, 256, 2, 2>(a, post, att, stream) : launch_attend_tail_as<T, 256, 4, 2>(a, post, att, stream);
  return half ? launch_attend_tail_as<T, 512, 2, 2>(a, post, att, stream) : hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_attend_tail(const moda_hip_block_tail_args* t, const KArgs& att, hipStream_t stream) {
  const TailArgs a = tail_args(t);
  const bool post = t->post_norm != 0;
  return t->dtype == 0 ? launch_attend_tail_of<BF16>(a, post, att, stream) : launch_attend_tail_of<FP16>(a, post, att, stream);
}

}  // namespace moda
