// The bf16 kernels of the fused backward (a source of their own: they take long to compile).
#include "mdcn_backward_fused.h"

namespace mdcn {

template <>
void launch_fused<bf16_t>(const BwdFusedArgs &a, int ch, hipStream_t st) {
  launch_fused_impl<bf16_t>(a, ch, st);
}

}  // namespace mdcn
