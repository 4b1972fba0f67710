// gemm_mid_kernel for W4A16 (g.kil: the staged operand layout).
#include "gemm_mid.h"

hipError_t ic_launch_mid_w16(const ic_gemm::GemmArgs& g, int tile, int S, hipStream_t st) {
  return g.kil ? launch_mid<big::W16, true>(g, tile, S, st) : launch_mid<big::W16, false>(g, tile, S, st);
}
