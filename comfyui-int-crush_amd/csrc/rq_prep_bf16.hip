// Fast-path preparation kernels for bf16 activations without quantization
// (ic_prepare_activation): the prepared row leaves in the activation type.
// Rows with either SmoothRot factors or a perm, and those with neither, here;
// rows with both in rq_prep_bf16_both.hip.
#include "rq_fast.h"

hipError_t ic_rq_prep_bf16(const ic_rotq_args& a, hipStream_t st) {
  if (a.sr_rcp != nullptr && a.perm != nullptr) return ic_rq_prep_bf16_both(a, st);
  if (a.sr_rcp == nullptr && a.perm == nullptr) return launch_fast<IC_DTYPE_BF16, kRqPlain, 0, false>(a, st);
  return launch_fast<IC_DTYPE_BF16, kRqGeneral, 0, false>(a, st);
}
