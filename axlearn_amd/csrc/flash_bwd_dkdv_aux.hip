// The dK / dV kernel's instantiations with a dense bias and / or a dropout mask: one per combination of the
// two, with and without segment ids, leaving dS for the streaming dQ kernel or not (a bf16 bias alone:
// flash_bwd_dkdv_bias.hip).
#include "flash_bwd_dkdv_kernel.h"

namespace axl {

template <typename E, int D, bool HAS_SEG, int AUX>
static hipError_t launch_form(const BwdArgs& a, hipStream_t stream) {
  if (a.splits > 1) return a.ds ? launch_one<E, D, HAS_SEG, AUX, true, D, true>(a, stream) : launch_one<E, D, HAS_SEG, AUX, false, D, true>(a, stream);
  return a.ds ? launch_one<E, D, HAS_SEG, AUX, true, D, false>(a, stream) : launch_one<E, D, HAS_SEG, AUX, false, D, false>(a, stream);
}

template <typename E, int D, int AUX>
static hipError_t launch_mode(const BwdArgs& a, hipStream_t stream) {
  return a.seg ? launch_form<E, D, true, AUX>(a, stream) : launch_form<E, D, false, AUX>(a, stream);
}

template <typename E, int D>
static hipError_t launch_for(const BwdArgs& a, hipStream_t stream) {
  const int bias = a.aux.bias ? (a.aux.bias_f32 ? kAuxBias32 : kAuxBias16) : 0;
  switch (bias | (a.aux.drop ? kAuxDrop : 0)) {
    case kAuxBias16:  // beside segment ids
      return launch_form<E, D, true, kAuxBias16>(a, stream);
    case kAuxBias32: return launch_mode<E, D, kAuxBias32>(a, stream);
    case kAuxDrop: return launch_mode<E, D, kAuxDrop>(a, stream);
    case kAuxBias16 | kAuxDrop: return launch_mode<E, D, kAuxBias16 | kAuxDrop>(a, stream);
    default: return launch_mode<E, D, kAuxBias32 | kAuxDrop>(a, stream);
  }
}

hipError_t launch_bwd_dkdv_aux(const BwdArgs& a, int dtype, int head_dim, hipStream_t stream) {
  if (a.aux.bias && !a.aux.bias_f32 && !a.aux.drop && !a.seg) return launch_bwd_dkdv_bias(a, dtype, head_dim, stream);
  if (dtype == AXL_F16) return head_dim == 128 ? launch_for<ElemF16, 128>(a, stream) : launch_for<ElemF16, 64>(a, stream);
  return head_dim == 128 ? launch_for<ElemBf16, 128>(a, stream) : launch_for<ElemBf16, 64>(a, stream);
}

}  // namespace axl
