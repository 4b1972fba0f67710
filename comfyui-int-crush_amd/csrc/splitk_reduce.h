// Second kernel of the split-K launches with 16-bit outputs.
#pragma once
#include "ic_common.h"

namespace {

// Adds the K-slice partials in slice order and finishes the outputs as the
// unsplit epilogue does.  Bound by the partials' reads: four columns per
// thread (N and ldc multiples of 4, C 8-byte and ws 16-byte aligned) make them
// 16-byte loads.  512 x 3072 x 12288 W4A8 in two slices with a residual: this
// kernel 7.4 -> 6.2 us, both kernels 45.7 -> 44.4.  KIND 0: int32 sums and
// per-row scales (1: of 16 * q weights), 2: fp32 folds of groups, 3: fp32 sums
// (W4A16).
template <int KIND, int OUT_DT>
__global__ __launch_bounds__(256) void splitk_reduce4_kernel(
    const int32_t* __restrict__ ws, int S, const float* __restrict__ s_a, const float* __restrict__ s_w,
    const void* __restrict__ bias, int bias_dt, void* __restrict__ C, int64_t ldc, int M, int N, ic_epi epi) {
  const int64_t MN = (int64_t)M * N;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);
  float v[4];
  if constexpr (KIND < 2) {
    v4i t = *(const v4i*)(ws + i);
    for (int s = 1; s < S; ++s) t = t + *(const v4i*)(ws + s * MN + i);
    const float sa = s_a[m];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float a = (float)t[k];
      if constexpr (KIND == 1) a *= 0.0625f;
      v[k] = a * (sa * s_w[n + k]);
    }
  } else {
    v4f t = *(const v4f*)((const float*)ws + i);
    for (int s = 1; s < S; ++s) {
      const v4f u = *(const v4f*)((const float*)ws + s * MN + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) t[k] = t[k] + u[k];
    }
    const float sa = KIND == 2 ? s_a[m] : 1.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = KIND == 2 ? t[k] * sa : t[k];
  }
  u16 h[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (bias != nullptr) v[k] = v[k] + ld_any_f32(bias, bias_dt, n + k);
    v[k] = epi_apply(v[k], epi, m, n + k);
    h[k] = OUT_DT == IC_DTYPE_F16 ? f32_to_f16(v[k]) : f32_to_bf16(v[k]);
  }
  *(v2u*)((u16*)C + (int64_t)m * ldc + n) =
      v2u{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
}

}  // namespace
