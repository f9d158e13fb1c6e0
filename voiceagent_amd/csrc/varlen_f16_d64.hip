// F16 head_dim 64 instantiations of the varlen attention kernel (varlen_kernel.h).
#include "varlen_kernel.h"

namespace va {

template <>
bool launch_varlen_d<false, 64>(int G, const VarlenParams& p, bool causal, int64_t items_per_xcd,
                          hipStream_t st) {
  return dispatch_varlen_g<false, 64>(G, p, causal, items_per_xcd, st);
}

}  // namespace va
