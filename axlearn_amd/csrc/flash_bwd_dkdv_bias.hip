// The dK / dV kernel's instantiations with a bf16 bias and nothing else.
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

template <typename E, int D>
static hipError_t launch_for(const BwdArgs& a, hipStream_t stream) {
  return a.ds ? launch_one<E, D, false, kAuxBias16, true>(a, stream) : launch_one<E, D, false, kAuxBias16>(a, stream);
}

hipError_t launch_bwd_dkdv_bias(const BwdArgs& a, int dtype, int head_dim, hipStream_t stream) {
  if (dtype == AXL_F16) return head_dim == 128 ? launch_for<ElemF16, 128>(a, stream) : launch_for<ElemF16, 64>(a, stream);
  return head_dim == 128 ? launch_for<ElemBf16, 128>(a, stream) : launch_for<ElemBf16, 64>(a, stream);
}

}  // namespace axl
