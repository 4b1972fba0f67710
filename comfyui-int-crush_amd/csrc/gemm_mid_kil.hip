// gemm_mid_kernel on packed INT4 weights in the K-interleaved order.
#include "gemm_mid.h"

hipError_t ic_launch_mid_kil(const ic_gemm::GemmArgs& g, int mode, int tile, int S, hipStream_t st) {
  switch (mode) {
    case big::G128: return launch_mid<big::G128, true>(g, tile, S, st);
    case big::G64: return launch_mid<big::G64, true>(g, tile, S, st);
    case big::G32: return launch_mid<big::G32, true>(g, tile, S, st);
    case big::ROW4: return launch_mid<big::ROW4, true>(g, tile, S, st);
  }
  return hipErrorInvalidValue;
}
