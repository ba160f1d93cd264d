// Backward, query side: the preprocess kernel (-delta = -rowsum(o * do), moda_v14.py:525-539) and the
// dQ kernel (moda_v14.py:542-871, moda_v16.py:936-1220, fda_v12.py:432-638,
// fla/ops/attn/parallel.py:165-296).
//
// Same streaming structure as the forward kernel: a workgroup owns 32 query rows per wave
// (256 in the throughput launch shape, 64 or 128 in the small one) and streams 64-column K/V tiles
// (sequence keys, then the rows' depth slots) through an LDS ring.  The products run on the 16x16x32
// matrix instruction, which moves a quarter of the accumulator bits per multiply-add of the 32x32x16
// one and draws less power on a matrix pipe whose clock the power limit sets (measured on the
// long-sequence workload: about 9 % less time for the same tiles).  A wave's 32 rows are two 16-row
// blocks; lane (n, q) owns rows 16*nb + n and, inside a 16-column score block, columns slot_base(q) .. +3.
// P^T is recomputed from the saved base-2 LSE, dS^T = P^T * (dP^T - delta) is packed straight into the
// B operand of dQ^T += K^T * dS^T, K^T coming from the LDS transpose read of the K tile.
#include <type_traits>

#include "bwd_dq.h"
#include "geometry.h"
#include "kargs.h"
#include "tile.h"
#include "tile16.h"
#include "tuning.h"

namespace moda {

template <typename T, int HD>
__global__ __launch_bounds__(256) void delta_kernel(const KArgs a_in) {
  constexpr int TPR = HD / 8;         // threads per row
  constexpr int RPB = 256 / TPR;      // rows per block
  const int tid = threadIdx.x;
  // one-dimensional grid (row blocks of the longest sequence x batch*heads): the y extent of a grid stops at 65535
  const int nrb = (a_in.Tq + RPB - 1) / RPB;
  const int bh = blockIdx.x / nrb;
  const int rb = blockIdx.x - bh * nrb;
  KArgs a = a_in;
  int b = bh / a.Hq;
  const int hq = bh % a.Hq;
  enter_sequence(a, b);
  const int r = rb * RPB + tid / TPR;
  const int c = (tid % TPR) * 8;
  float acc = 0.f;
  if (r < a.Tq && c < a.Dv) {
    const uint16_t* op = a.o + b * a.so.b + hq * a.so.h + (int64_t)r * a.so.t + c;
    const uint16_t* dp = a.d_o + b * a.sdo.b + hq * a.sdo.h + (int64_t)r * a.sdo.t + c;
    const typename T::vec8 ov = *reinterpret_cast<const typename T::vec8*>(op);
    const typename T::vec8 dv = *reinterpret_cast<const typename T::vec8*>(dp);
#pragma unroll
    for (int i = 0; i < 8; i++) acc += (float)ov[i] * (float)dv[i];
  }
#pragma unroll
  for (int s = TPR / 2; s > 0; s >>= 1) acc += __shfl_xor(acc, s, 64);
  if (r < a.Tq && (tid % TPR) == 0) a.delta[((int64_t)b * a.Hq + hq) * a.delta_pitch + r] = -acc;
}

template <typename T, int HD>
hipError_t launch_delta_t(const KArgs& a, hipStream_t stream) {
  if (a.Tq == 0 || a.B * a.Hq == 0) return hipSuccess;
  constexpr int RPB = 256 / (HD / 8);
  const int64_t nblk = delta_kernel_blocks(a, RPB);
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((delta_kernel<T, HD>), dim3((unsigned)nblk), dim3(256), 0, stream, a);
  return hipGetLastError();
}

template <typename T, int HD, typename Shape, int ADDR>
hipError_t launch_dq_t_shape(const KArgs& a, hipStream_t stream) {
  constexpr size_t smem = dq_lds<HD, Shape, ADDR>();
  static LdsAttrState attr;
  const hipError_t ea = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&dq_kernel<T, HD, Shape, ADDR>), smem);
  if (ea != hipSuccess) return ea;
  constexpr int rows = 16 * Shape::NB * Shape::W;
  const int64_t nblk = row_kernel_blocks(a, rows);
  if (nblk == 0) return hipSuccess;
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((dq_kernel<T, HD, Shape, ADDR>), dim3((unsigned)nblk), dim3(64 * Shape::W), smem, stream, a);
  return hipGetLastError();
}

template <typename T, int HD, int ADDR>
hipError_t launch_dq_t_addr(const KArgs& a, bool small, hipStream_t stream) {
  if constexpr (HD <= 64) {
    const ShortRows rows = (ADDR & 3) ? ShortRows::kNone : pick_short_rows(a.Tq, (long long)a.B * a.Hq, a.causal, a.compute_units);
    if (rows == ShortRows::kTwoStages) return launch_dq_t_shape<T, HD, RowShort, ADDR & ~3>(a, stream);
    if (rows == ShortRows::kThreeStages) return launch_dq_t_shape<T, HD, RowShort3, ADDR & ~3>(a, stream);
    return launch_dq_t_shape<T, HD, RowSmall<HD>, ADDR>(a, stream);
  } else if constexpr (HD > 128) {
    return launch_dq_t_shape<T, HD, RowWide, ADDR>(a, stream);  // one shape for the wide tiles
  } else {
    if (small && !(ADDR & 1)) return launch_dq_t_shape<T, HD, RowSmall<HD>, ADDR & ~1>(a, stream);  // slices wider than 2 GiB: never small
    return launch_dq_t_shape<T, HD, RowLarge, ADDR>(a, stream);
  }
}

template <typename T, int HD>
hipError_t launch_dq_t(const KArgs& a, hipStream_t stream) {
  const bool wide = !narrow_slices(a);
  const bool small = a.cu ? use_small_rows(a.delta_pitch, a.Hq, a.compute_units)  // the rows there are, not those of the grid
                          : use_small_rows(a.Tq, (long long)a.B * a.Hq, a.compute_units);
  switch ((wide ? 1 : 0) | (a.cu ? 2 : 0) | (a.L == 0 ? 4 : 0) | (a.L > 0 && a.Lv != a.L ? 8 : 0)) {
    case 0: return launch_dq_t_addr<T, HD, 0>(a, small, stream);
    case 1: return launch_dq_t_addr<T, HD, 1>(a, small, stream);
    case 2: return launch_dq_t_addr<T, HD, 2>(a, small, stream);
    case 3: return launch_dq_t_addr<T, HD, 3>(a, small, stream);
    case 4: return launch_dq_t_addr<T, HD, 4>(a, small, stream);
    case 5: return launch_dq_t_addr<T, HD, 5>(a, small, stream);
    case 6: return launch_dq_t_addr<T, HD, 6>(a, small, stream);
    case 7: return launch_dq_t_addr<T, HD, 7>(a, small, stream);
    case 8: return launch_dq_t_addr<T, HD, 8>(a, small, stream);
    case 9: return launch_dq_t_addr<T, HD, 9>(a, small, stream);
    case 10: return launch_dq_t_addr<T, HD, 10>(a, small, stream);
    default: return launch_dq_t_addr<T, HD, 11>(a, small, stream);
  }
}

hipError_t launch_delta(const KArgs& a, int dtype, int hd, hipStream_t stream) {
  if (dtype == 0 && hd == 128) return launch_delta_t<BF16, 128>(a, stream);
  if (dtype == 0 && hd == 64) return launch_delta_t<BF16, 64>(a, stream);
  if (dtype == 1 && hd == 128) return launch_delta_t<FP16, 128>(a, stream);
  if (dtype == 1 && hd == 64) return launch_delta_t<FP16, 64>(a, stream);
  if (dtype == 0 && hd == 256) return launch_delta_t<BF16, 256>(a, stream);
  if (dtype == 1 && hd == 256) return launch_delta_t<FP16, 256>(a, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_dq(const KArgs& a, int dtype, int hd, hipStream_t stream) {
  if (dtype == 0 && hd == 128) return launch_dq_t<BF16, 128>(a, stream);
  if (dtype == 0 && hd == 64) return launch_dq_t<BF16, 64>(a, stream);
  if (dtype == 1 && hd == 128) return launch_dq_t<FP16, 128>(a, stream);
  if (dtype == 1 && hd == 64) return launch_dq_t<FP16, 64>(a, stream);
  if (dtype == 0 && hd == 256) return launch_dq_t<BF16, 256>(a, stream);
  if (dtype == 1 && hd == 256) return launch_dq_t<FP16, 256>(a, stream);
  return hipErrorInvalidValue;
}

}  // namespace moda
