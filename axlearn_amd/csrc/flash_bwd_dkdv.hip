// The dK / dV kernel's plain instantiations (no dense bias, no dropout mask) and its launcher.
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

template <typename E, int D, bool SPILL>
static hipError_t launch_plain(const BwdArgs& a, hipStream_t stream) {
  return a.seg ? launch_one<E, D, true, 0, SPILL>(a, stream) : launch_one<E, D, false, 0, SPILL>(a, stream);
}

template <typename E>
static hipError_t launch_for(const BwdArgs& a, int head_dim, hipStream_t stream) {
  if (a.ds) return head_dim == 128 ? launch_plain<E, 128, true>(a, stream) : launch_plain<E, 64, true>(a, stream);
  return head_dim == 128 ? launch_plain<E, 128, false>(a, stream) : launch_plain<E, 64, false>(a, stream);
}

hipError_t launch_bwd_dkdv(const BwdArgs& a, int dtype, int head_dim, bool aux, hipStream_t stream) {
  if (aux) return launch_bwd_dkdv_aux(a, dtype, head_dim, stream);
  return dtype == AXL_F16 ? launch_for<ElemF16>(a, head_dim, stream) : launch_for<ElemBf16>(a, head_dim, stream);
}

}  // namespace axl
