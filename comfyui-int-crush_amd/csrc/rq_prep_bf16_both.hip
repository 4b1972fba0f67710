// Fast-path preparation kernels for bf16 activations without quantization, with
// both SmoothRot factors and a perm.
#include "rq_fast.h"

hipError_t ic_rq_prep_bf16_both(const ic_rotq_args& a, hipStream_t st) {
  return launch_fast<IC_DTYPE_BF16, kRqBoth, 0, false>(a, st);
}
