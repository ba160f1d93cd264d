// dQ and sequence dK/dV of small problems on the 64-wide tiles in one launch: the workgroups of dq_kernel and of
// dkv_flat_kernel side by side.  Where both together do not fill the machine, each launch is a chain of a few dependent
// tiles behind its own start and end; together they take as long as the longer one.  The dK/dV workgroups form the row sums
// of o * do themselves (OWN_DELTA).  2 x 95 tokens, four heads of two query rows, eight slots, fp16: 25.6 -> 19.8
// us of kernels and a launch less, the replayed training step 35.0 -> 29.3 us; 8 x 197 tokens, six heads, twelve slots 71.1 -> 64.2.
#define MODA_SIDE_BY_SIDE
#include "bwd_dkv_flat.h"
#include "bwd_dq.h"

namespace moda {

template <typename T, int ADDR>
__global__ __launch_bounds__(256, 2) void bwd_short_kernel(const KArgs a, int row_blocks) {
  static_assert(16 * RowSmall<64>::NB * RowSmall<64>::W == kBwdShortRows, "the grid's rows are the workgroup's");
  if ((int)blockIdx.x < row_blocks)
    dq_body<T, 64, RowSmall<64>, ADDR>(a, blockIdx.x);
  else
    dkv_flat_body<T, 64, false, false, 4, true>(a, (int)blockIdx.x - row_blocks);
}

template <typename T, int ADDR>
hipError_t launch_short_t(const KArgs& a, hipStream_t stream) {
  constexpr size_t lds_dq = dq_lds<64, RowSmall<64>, ADDR>(), lds_dkv = dkv_flat_lds<64, 4, true>();
  constexpr size_t smem = lds_dq > lds_dkv ? lds_dq : lds_dkv;
  static_assert(2 * smem <= 160 * 1024, "two workgroups a compute unit");
  static LdsAttrState attr;
  const hipError_t ea = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&bwd_short_kernel<T, ADDR>), smem);
  if (ea != hipSuccess) return ea;
  const int64_t columns = dkv_flat_blocks(a, 32), rows = row_kernel_blocks(a, kBwdShortRows);
  hipLaunchKernelGGL((bwd_short_kernel<T, ADDR>), dim3((unsigned)(columns + rows)), dim3(256), smem, stream, a, (int)rows);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_short_as(const KArgs& a, hipStream_t stream) {
  if (a.L == 0) return launch_short_t<T, 4>(a, stream);
  return a.Lv != a.L ? launch_short_t<T, 8>(a, stream) : launch_short_t<T, 0>(a, stream);
}

// dtype: 0 bf16, 1 fp16; the caller asks bwd_one_launch first
hipError_t launch_bwd_short(const KArgs& a, int dtype, hipStream_t stream) {
  return dtype == 0 ? launch_short_as<BF16>(a, stream) : launch_short_as<FP16>(a, stream);
}

}  // namespace moda
