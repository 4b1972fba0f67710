// gemm_mid_kernel on int8 weights (per-row scales, or INT4 unpacked to bytes with group scales).
#include "gemm_mid.h"

hipError_t ic_launch_mid_i8(const ic_gemm::GemmArgs& g, int mode, int tile, int S, hipStream_t st) {
  switch (mode) {
    case big::ROW8: return launch_mid<big::ROW8, false>(g, tile, S, st);
    case big::G128I8: return launch_mid<big::G128I8, false>(g, tile, S, st);
  }
  return hipErrorInvalidValue;
}
