// The dK / dV kernel's plain instantiations (no dense bias, no dropout mask) and its launcher.
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

template <typename E, int D, bool SPILL, int W = D>
static hipError_t launch_plain(const BwdArgs& a, hipStream_t stream) {
  return a.seg ? launch_one<E, D, true, 0, SPILL, W>(a, stream) : launch_one<E, D, false, 0, SPILL, W>(a, stream);
}

template <typename E>
static hipError_t launch_for(const BwdArgs& a, int head_dim, hipStream_t stream) {
  if (head_dim == 96) return a.ds ? launch_plain<E, 128, true, 96>(a, stream) : launch_plain<E, 128, false, 96>(a, stream);
  if (a.ds) return head_dim == 128 ? launch_plain<E, 128, true>(a, stream) : launch_plain<E, 64, true>(a, stream);
  return head_dim == 128 ? launch_plain<E, 128, false>(a, stream) : launch_plain<E, 64, false>(a, stream);
}

template <typename E>
static hipError_t launch_sum(const BwdArgs& a, int head_dim, hipStream_t stream) {
  const dim3 grid(a.S / 32 * a.B * a.Hkv, 2);
  if (head_dim == 128) hipLaunchKernelGGL((flash_bwd_dkdv_combine_kernel<E, 128>), grid, dim3(256), 0, stream, a);
  else if (head_dim == 96) hipLaunchKernelGGL((flash_bwd_dkdv_combine_kernel<E, 96>), grid, dim3(192), 0, stream, a);
  else hipLaunchKernelGGL((flash_bwd_dkdv_combine_kernel<E, 64>), grid, dim3(128), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv(const BwdArgs& a, int dtype, int head_dim, bool aux, hipStream_t stream) {
  hipError_t err;
  if (aux) err = launch_bwd_dkdv_aux(a, dtype, head_dim, stream);
  else err = dtype == AXL_F16 ? launch_for<ElemF16>(a, head_dim, stream) : launch_for<ElemBf16>(a, head_dim, stream);
  if (err != hipSuccess || a.splits <= 1) return err;
  return dtype == AXL_F16 ? launch_sum<ElemF16>(a, head_dim, stream) : launch_sum<ElemBf16>(a, head_dim, stream);
}

}  // namespace axl
