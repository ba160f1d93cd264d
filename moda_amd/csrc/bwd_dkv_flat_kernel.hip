// Launches of the sequence dK/dV on the 64-wide tiles (bwd_dkv_flat.h).
#include "bwd_dkv_flat.h"

namespace moda {

template <typename T, int HD, bool VARLEN, bool SPLIT, int RW = 1>
hipError_t launch_dkv_flat_t(const KArgs& a, hipStream_t stream) {
  constexpr size_t smem = dkv_flat_lds<HD, RW, false>();
  static LdsAttrState attr;
  const hipError_t ea = allow_dynamic_lds(attr, reinterpret_cast<const void*>(&dkv_flat_kernel<T, HD, VARLEN, SPLIT, RW>), smem);
  if (ea != hipSuccess) return ea;
  const int64_t nblk = dkv_flat_blocks(a, 128 / RW, SPLIT ? a.dkv_split : 1);
  if (nblk == 0) return hipSuccess;
  if (nblk >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((dkv_flat_kernel<T, HD, VARLEN, SPLIT, RW>), dim3((unsigned)nblk), dim3(256), smem, stream, a);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_dkv_flat_as(const KArgs& a, hipStream_t stream) {
  const bool split = a.dkv_split > 1;
  if (a.cu) return split ? launch_dkv_flat_t<T, 64, true, true>(a, stream) : launch_dkv_flat_t<T, 64, true, false>(a, stream);
  if (dkv_flat_row_waves(a)) return launch_dkv_flat_t<T, 64, false, false, 4>(a, stream);
  return split ? launch_dkv_flat_t<T, 64, false, true>(a, stream) : launch_dkv_flat_t<T, 64, false, false>(a, stream);
}

// dtype: 0 bf16, 1 fp16; 64-wide tiles only (the caller asks takes_dkv_flat first)
hipError_t launch_dkv_flat(const KArgs& a, int dtype, hipStream_t stream) {
  return dtype == 0 ? launch_dkv_flat_as<BF16>(a, stream) : launch_dkv_flat_as<FP16>(a, stream);
}

}  // namespace moda
