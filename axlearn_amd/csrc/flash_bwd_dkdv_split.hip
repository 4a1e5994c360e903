// dK/dV of launches whose workgroups share the query tiles of a key block, no bias or a bf16 bias alone (the forms with
// other inputs are in flash_bwd_dkdv_aux.hip).
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

hipError_t launch_bwd_dkdv_split(const BwdArgs& a, int dtype, int head_dim, hipStream_t stream) {
  return dtype == AXL_F16 ? launch_plain_width<ElemF16, true>(a, head_dim, stream) : launch_plain_width<ElemBf16, true>(a, head_dim, stream);
}

hipError_t launch_bwd_dkdv_split_bias(const BwdArgs& a, int dtype, int head_dim, hipStream_t stream) {
  if (dtype == AXL_F16) return head_dim == 128 ? launch_bias<ElemF16, true, 128>(a, stream) : launch_bias<ElemF16, true, 64>(a, stream);
  return head_dim == 128 ? launch_bias<ElemBf16, true, 128>(a, stream) : launch_bias<ElemBf16, true, 64>(a, stream);
}

}  // namespace axl
