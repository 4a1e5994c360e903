// The dK / dV kernel's plain instantiations (no dense bias, no dropout mask) and its launcher.
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

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
  else if (a.splits > 1) err = launch_bwd_dkdv_split(a, dtype, head_dim, stream);
  else if (dtype == AXL_F16) err = launch_plain_width<ElemF16, false>(a, head_dim, stream);
  else err = launch_plain_width<ElemBf16, false>(a, head_dim, stream);
  if (err != hipSuccess || a.splits <= 1) return err;
  return dtype == AXL_F16 ? launch_sum<ElemF16>(a, head_dim, stream) : launch_sum<ElemBf16>(a, head_dim, stream);
}

}  // namespace axl
