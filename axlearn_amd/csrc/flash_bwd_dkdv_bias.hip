// The dK / dV kernel's instantiations with a bf16 bias and nothing else.
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

hipError_t launch_bwd_dkdv_bias(const BwdArgs& a, int dtype, int head_dim, hipStream_t stream) {
  if (a.splits > 1) return launch_bwd_dkdv_split_bias(a, dtype, head_dim, stream);
  if (dtype == AXL_F16) return head_dim == 128 ? launch_bias<ElemF16, false, 128>(a, stream) : launch_bias<ElemF16, false, 64>(a, stream);
  return head_dim == 128 ? launch_bias<ElemBf16, false, 128>(a, stream) : launch_bias<ElemBf16, false, 64>(a, stream);
}

}  // namespace axl
