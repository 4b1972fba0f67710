// INT8-MFMA and W4A16 GEMM on small output tiles (gfx950), for launches whose
// 256-row tiles would leave most CUs idle or multiply padding: 17 to a few
// hundred tokens, narrow outputs, long K.
//
// A 256-thread workgroup of 2 x 2 waves owns a (32 TM) x (32 TN) tile, each
// wave TM x TN blocks of v_mfma_i32_16x16x64_i8 (v_mfma_f32_16x16x32 for
// W4A16).  The weight modes, their arithmetic and their fragment layouts are
// those of gemm_i8_big_kernel (per-group folds of exact int32 sums in K
// order, per-row int32 sums, or fp32 sums of dequantized weights), so every
// unsplit result is the same bit for bit for the INT8 modes.
//
// What bounds it: few tiles are in flight, so a stage costs its latency (DMA,
// barrier, LDS reads) before its work.  Hence two or three workgroups share a
// CU, each with its own barrier and an NS-slot DMA ring (NS - 1 stages in
// flight), and one covers the other's waits; the large tiles run one
// workgroup of eight waves per CU in lockstep.  Each stage has one barrier:
// the slot filled next is the one every wave finished before it.
//
// PART (split-K): workgroup (x, y) computes K slice y of gridDim.y and writes
// 4-byte partials (int32 sums, or the fp32 fold) to
// ws[(y * M + m) * N + n]; splitk_reduce4_kernel adds them in slice order.
#pragma once
#include <type_traits>

#include "gemm_i8_big.h"
#include "gemm_mid_plan.h"
#include "splitk_reduce.h"

namespace {
namespace mid {
constexpr int kMT = 256;  // threads per workgroup
using big::G128;
using big::G128I8;
using big::G32;
using big::G64;
using big::ROW4;
using big::ROW8;
using big::W16;

template <int TM_, int TN_, int NS_, int MODE_>
struct Cfg {
  static constexpr int TM = TM_, TN = TN_, NS = NS_, MODE = MODE_;
  static constexpr bool GROUPED = MODE <= G64 || MODE == G32 || MODE == G128I8;
  static constexpr bool F64 = MODE == G64, F32 = MODE == G32, DEQ = MODE == W16;
  static constexpr bool INT8W = MODE == ROW8 || MODE == G128I8;
  static constexpr bool SCALED = GROUPED || DEQ;
  static constexpr int BM = 32 * TM, BN = 32 * TN, WROWS = 16 * TM, WCOLS = 16 * TN;
  static constexpr int KS = DEQ ? 64 : kBK;             // K values per stage
  static constexpr int NSC = F32 ? 4 : (F64 ? 2 : 1);   // scale rows per stage
  static constexpr int A_BYTES = BM * kBK;
  static constexpr int B_BYTES = INT8W ? BN * kBK : BN * KS / 2;
  static constexpr int S_BYTES = BN * 4, S_WAVES = BN / 64;
  static constexpr int SLOT = A_BYTES + B_BYTES + (SCALED ? NSC * S_BYTES : 0);
  static constexpr int A_BLOCKS = BM / 8, A_PER = (A_BLOCKS + 3) / 4;       // 1 KB DMA blocks, per wave
  static constexpr int B_BLOCKS = B_BYTES / 1024, B_PER = (B_BLOCKS + 3) / 4;
  static constexpr int EPI_RS = BN + 8;
  static constexpr size_t epi_bytes = (size_t)BM * EPI_RS * 2 + (size_t)(BM + 2 * BN) * 4;
  static constexpr size_t lds_bytes = (size_t)NS * SLOT > epi_bytes ? (size_t)NS * SLOT : epi_bytes;
  static_assert(BN % 64 == 0 && SLOT % 16 == 0 && lds_bytes <= 80 * 1024, "two workgroups per CU");
  static_assert(BM <= kMT && BN <= kMT, "one epilogue operand per thread");
};

// Block until at most n vector-memory operations are outstanding (n is
// wave-uniform; at most MAXN).
template <int MAXN> IC_DEV void wait_vm_upto(int n) {
  if constexpr (MAXN == 0) {
    wait_vm<0>();
  } else {
    if (n >= MAXN) wait_vm<MAXN>();
    else wait_vm_upto<MAXN - 1>(n);
  }
}
}  // namespace mid

// KIL: packed INT4 in the K-interleaved order, or (W16) the staged operand
// layout, as in gemm_i8_big_kernel.
template <class CF, int OUT_DT, bool EPI, bool KIL, bool PART>
__global__ __launch_bounds__(mid::kMT, 2) void gemm_mid_kernel(
    const int8_t* __restrict__ A, int64_t lda, const uint8_t* __restrict__ B, int64_t ldb,
    const float* __restrict__ s_a, const float* __restrict__ s_w, int G, const void* __restrict__ bias, int bias_dt,
    void* __restrict__ C, int64_t ldc, int M, int N, int K, int32_t* __restrict__ ws, ic_epi epi) {
  using namespace mid;
  constexpr int TM = CF::TM, TN = CF::TN, NS = CF::NS, LA = NS - 1, BM = CF::BM, BN = CF::BN, SLOT = CF::SLOT;
  constexpr int A_BYTES = CF::A_BYTES, B_BYTES = CF::B_BYTES, S_BYTES = CF::S_BYTES, KS = CF::KS;
  constexpr bool GROUPED = CF::GROUPED, F64 = CF::F64, F32 = CF::F32, DEQ = CF::DEQ, INT8W = CF::INT8W;
  constexpr bool STAGED = DEQ && KIL;
  static_assert(OUT_DT != IC_DTYPE_F32 && !(KIL && INT8W) && !(EPI && DEQ), "mid tile modes");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  // epilogue operands, loaded now so that their latency passes under the loop
  float pre_sa = 0.0f, pre_b = 0.0f, pre_sw = 0.0f;
  if constexpr (!PART) {
    if (!DEQ && tid < BM) pre_sa = s_a[min(m0 + tid, M - 1)];
    if (tid < BN && bias != nullptr) pre_b = ld_any_f32(bias, bias_dt, min(n0 + tid, N - 1));
    if (!GROUPED && !DEQ && tid < BN) pre_sw = s_w[min(n0 + tid, N - 1)];
  }
  const int KT_all = K / KS;
  const int kt0 = PART ? (int)((int64_t)blockIdx.y * KT_all / gridDim.y) : 0;
  const int KT = PART ? (int)((int64_t)(blockIdx.y + 1) * KT_all / gridDim.y) - kt0 : KT_all;
  // scale blocks (of 128, 64 or 32 columns) per group
  const int bpg = (K / G) / (F32 ? 32 : (F64 || DEQ ? 64 : kBK));

  // ---- DMA addressing, as in gemm_i8_big_kernel (rows past M or N re-read the last)
  uint32_t a_off[CF::A_PER], b_off[CF::B_PER];
#pragma unroll
  for (int c = 0; c < CF::A_PER; ++c) {
    const int row = 8 * (wave + 4 * c) + (lane >> 3);
    a_off[c] = (uint32_t)(min(row, M - 1 - m0) * lda + (((lane & 7) ^ swz(row)) << 4));
  }
#pragma unroll
  for (int c = 0; c < CF::B_PER; ++c) {
    const int blk = wave + 4 * c;
    if constexpr (INT8W) {
      const int row = 8 * blk + (lane >> 3);
      b_off[c] = (uint32_t)(min(row, N - 1 - n0) * ldb + (((lane & 7) ^ swz(row)) << 4));
    } else if constexpr (DEQ) {
      const int row = 32 * blk + (lane >> 1);
      b_off[c] = (uint32_t)(min(row, N - 1 - n0) * (STAGED ? 32 : ldb) + (((lane & 1) ^ ((row >> 3) & 1)) << 4));
    } else {
      const int row = 16 * blk + (lane >> 2);
      b_off[c] = (uint32_t)(min(row, N - 1 - n0) * ldb + (((lane & 3) ^ ((lane >> 4) & 3)) << 4));
    }
  }
  // scales: from the last waves, which issue no more activation or weight DMAs than the others
  const int sw_id = wave - (4 - (STAGED ? 1 : CF::S_WAVES));
  const bool s_wave = CF::SCALED && sw_id >= 0;
  const uint32_t s_off = STAGED ? (uint32_t)(min(4 * lane, N - 4 - n0) * 4)
                                : (uint32_t)(min(64 * max(sw_id, 0) + lane, N - 1 - n0) * G * 4);
  const int8_t* a_base = A + (int64_t)m0 * lda + (int64_t)kt0 * kBK;
  const uint8_t* b_base =
      B + (int64_t)n0 * (STAGED ? 32 : ldb) + (int64_t)kt0 * (INT8W ? kBK : (STAGED ? ldb : KS / 2));
  const float* s_base = s_w + (int64_t)n0 * (STAGED ? 1 : G);
  auto issue = [&](int kt) {
    const uint32_t slot = lds0 + (uint32_t)((kt % NS) * SLOT);
    if (s_wave) {
      const uint32_t sl = slot + (uint32_t)(A_BYTES + B_BYTES + sw_id * 256);
      const int g = kt0 + kt;
      if constexpr (STAGED) {
        if (lane < BN / 4) dma16(s_off, s_base + (int64_t)(g / bpg) * N, slot + (uint32_t)(A_BYTES + B_BYTES));
      } else {
#pragma unroll
        for (int h = 0; h < CF::NSC; ++h) dma4(s_off, s_base + (CF::NSC * g + h) / bpg, sl + (uint32_t)(h * S_BYTES));
      }
    }
#pragma unroll
    for (int c = 0; c < CF::B_PER; ++c) {
      const int blk = wave + 4 * c;
      if (blk < CF::B_BLOCKS)
        dma16(b_off[c], b_base + (int64_t)kt * (INT8W ? kBK : (STAGED ? ldb : KS / 2)),
              slot + (uint32_t)(A_BYTES + blk * 1024));
    }
#pragma unroll
    for (int c = 0; c < CF::A_PER; ++c) {
      const int blk = wave + 4 * c;
      if (blk < CF::A_BLOCKS) dma16(a_off[c], a_base + (int64_t)kt * kBK, slot + (uint32_t)(blk * 1024));
    }
  };
  int per_stage = s_wave ? (STAGED ? 1 : CF::NSC) : 0;  // this wave's DMAs per stage
#pragma unroll
  for (int c = 0; c < CF::B_PER; ++c) per_stage += wave + 4 * c < CF::B_BLOCKS;
#pragma unroll
  for (int c = 0; c < CF::A_PER; ++c) per_stage += wave + 4 * c < CF::A_BLOCKS;
  constexpr int kMaxPer = CF::A_PER + CF::B_PER + (CF::SCALED ? CF::NSC : 0);

  // ---- fragments (gemm_i8_big_kernel's layouts)
  const int fr_n = wc * CF::WCOLS + (lane & 15), fr_c = lane >> 4;
  const uint32_t fr0 = (uint32_t)(fr_n * 64 + 8 * (fr_c & 1) + (((fr_c >> 1) ^ ((fr_n >> 2) & 3)) << 4));
  const uint32_t fr1 = (uint32_t)(fr_n * 64 + 8 * (fr_c & 1) + (((2 + (fr_c >> 1)) ^ ((fr_n >> 2) & 3)) << 4));
  const uint32_t fq0 = (uint32_t)lds_off(fr_n, fr_c), fq1 = (uint32_t)lds_off(fr_n, 4 + fr_c);
  const uint32_t fw = (uint32_t)(fr_n * 32 + 4 * fr_c), fsw = (uint32_t)(((lane >> 3) & 1) << 4);
  const uint32_t fa0 = (uint32_t)lds_off(wr * CF::WROWS + (lane & 15), fr_c);
  const uint32_t fa1 = (uint32_t)lds_off(wr * CF::WROWS + (lane & 15), 4 + fr_c);

  using AccT = std::conditional_t<GROUPED || DEQ, v4f, v4i>;
  AccT acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = AccT{0, 0, 0, 0};

  auto stage = [&](int kt) {
    const char* sl = smem + (kt % NS) * SLOT;
    const char* sb = sl + A_BYTES;
    const float* sS = (const float*)(sb + B_BYTES) + wc * CF::WCOLS + (lane & 15);
    v4i b0[TN], b1[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (INT8W) {
        b0[j] = *(const v4i*)(sb + j * 16 * kBK + fq0);
        b1[j] = *(const v4i*)(sb + j * 16 * kBK + fq1);
      } else if constexpr (DEQ) {
        const uint32_t p0 = *(const uint32_t*)(sb + j * 16 * 32 + fw + fsw);
        const uint32_t p1 = *(const uint32_t*)(sb + j * 16 * 32 + fw + (16u ^ fsw));
        const DeqScale d = deq_scale<OUT_DT>(sS[16 * j]);
        uint32_t w[8];
        deq8<OUT_DT>(p0, d, w);
        deq8<OUT_DT>(p1, d, w + 4);
        b0[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        b1[j] = v4i{(int)w[4], (int)w[5], (int)w[6], (int)w[7]};
      } else {
        const v2u q0 = *(const v2u*)(sb + j * 16 * 64 + fr0);
        const v2u q1 = *(const v2u*)(sb + j * 16 * 64 + fr1);
        uint32_t w[8];
        if constexpr (KIL) {
          unpack8_x16_kil(q0.x, w[0], w[1]);
          unpack8_x16_kil(q0.y, w[2], w[3]);
          unpack8_x16_kil(q1.x, w[4], w[5]);
          unpack8_x16_kil(q1.y, w[6], w[7]);
        } else {
          unpack8_x16(q0.x, w[0], w[1]);
          unpack8_x16(q0.y, w[2], w[3]);
          unpack8_x16(q1.x, w[4], w[5]);
          unpack8_x16(q1.y, w[6], w[7]);
        }
        b0[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        b1[j] = v4i{(int)w[4], (int)w[5], (int)w[6], (int)w[7]};
      }
    }
    float sw[CF::NSC][TN];
    if constexpr (GROUPED) {
#pragma unroll
      for (int h = 0; h < CF::NSC; ++h)
#pragma unroll
        for (int j = 0; j < TN; ++j) sw[h][j] = sS[h * BN + 16 * j] * (INT8W ? 1.0f : 0.0625f);
    }
    // facc = fma(f32(block sum), s_w [/ 16], facc), blocks in K order
    auto fold = [&](AccT& f, const v4i& t, float s) {
#pragma unroll
      for (int r = 0; r < 4; ++r) f[r] = __builtin_fmaf((float)t[r], s, f[r]);
    };
    constexpr v4i z = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const v4i a0 = *(const v4i*)(sl + fa0 + i * 16 * kBK);
      const v4i a1 = *(const v4i*)(sl + fa1 + i * 16 * kBK);
      if constexpr (F32) {
        const bool lo = fr_c < 2;
        const v4i a0l = {lo ? a0[0] : 0, lo ? a0[1] : 0, lo ? a0[2] : 0, lo ? a0[3] : 0};
        const v4i a0h = {lo ? 0 : a0[0], lo ? 0 : a0[1], lo ? 0 : a0[2], lo ? 0 : a0[3]};
        const v4i a1l = {lo ? a1[0] : 0, lo ? a1[1] : 0, lo ? a1[2] : 0, lo ? a1[3] : 0};
        const v4i a1h = {lo ? 0 : a1[0], lo ? 0 : a1[1], lo ? 0 : a1[2], lo ? 0 : a1[3]};
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a0l, b0[j], z, 0, 0, 0), sw[0][j]);
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a0h, b0[j], z, 0, 0, 0), sw[1][j]);
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a1l, b1[j], z, 0, 0, 0), sw[2][j]);
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a1h, b1[j], z, 0, 0, 0), sw[3][j]);
        }
      } else if constexpr (F64) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0[j], z, 0, 0, 0), sw[0][j]);
          fold(acc[i][j], __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1[j], z, 0, 0, 0), sw[1][j]);
        }
      } else if constexpr (GROUPED) {
        v4i t[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) t[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0[j], z, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TN; ++j) t[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1[j], t[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TN; ++j) fold(acc[i][j], t[j], sw[0][j]);
      } else if constexpr (DEQ) {
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = big::mfma16<OUT_DT>(a0, b0[j], acc[i][j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = big::mfma16<OUT_DT>(a1, b1[j], acc[i][j]);
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1[j], acc[i][j], 0, 0, 0);
      }
    }
  };

  for (int s = 0; s < LA && s < KT; ++s) issue(s);
  for (int s = 0; s < KT; ++s) {
    // stage s has landed once only the DMAs of the stages after it remain
    wait_vm_upto<(LA - 1) * kMaxPer>(min(LA - 1, KT - 1 - s) * per_stage);
    lds_barrier();  // everyone's part of stage s; everyone is done with the slot filled next
    if (s + LA < KT) issue(s + LA);
    stage(s);
  }

  if constexpr (PART) {
    int32_t* p = ws + (int64_t)blockIdx.y * M * N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wr * CF::WROWS + 16 * i + 4 * fr_c + r, n = n0 + fr_n + 16 * j;
          if (m < M && n < N) {
            if constexpr (GROUPED || DEQ) ((float*)p)[(int64_t)m * N + n] = acc[i][j][r];
            else p[(int64_t)m * N + n] = acc[i][j][r];
          }
        }
    return;
  }

  // ---- epilogue: finish in registers, stage the tile row-major, store 16-byte runs
  constexpr int RS = CF::EPI_RS, CPR = BN / 8;
  lds_barrier();
  u16* ot = (u16*)smem;
  float* sa_l = (float*)(smem + BM * RS * 2);
  float* b_l = sa_l + BM;
  float* sw_l = b_l + BN;
  bool res_lds = false;
  if constexpr (EPI) {
    res_lds = epi.res != nullptr;
    if (res_lds) {
      for (int c = tid; c < BM * CPR; c += kMT) {
        const int row = c / CPR, col = (c % CPR) * 8, m = m0 + row, n = n0 + col;
        if (m < M && n < N)
          *(v4u*)(ot + row * RS + col) = *(const v4u*)((const u16*)epi.res + (int64_t)m * epi.ldr + n);
      }
    }
  }
  if (tid < BM) sa_l[tid] = pre_sa;
  if (tid < BN) {
    b_l[tid] = pre_b;
    sw_l[tid] = pre_sw;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int nl = fr_n + 16 * j;
    const float b = b_l[nl], sw = sw_l[nl];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ml = wr * CF::WROWS + 16 * i + 4 * fr_c + r;
        float v;
        if constexpr (GROUPED) {
          v = acc[i][j][r] * sa_l[ml];
        } else if constexpr (DEQ) {
          v = acc[i][j][r];
        } else {
          float a = (float)acc[i][j][r];
          if constexpr (!INT8W) a *= 0.0625f;
          v = a * (sa_l[ml] * sw);
        }
        if (bias != nullptr) v = v + b;
        if constexpr (EPI) {
          v = epi_act(v, epi.act);
          if (res_lds) {
            const u16 rv = ot[ml * RS + nl];
            v = v + (epi.res_dt == IC_DTYPE_F16 ? f16_to_f32(rv) : bf16_to_f32(rv));
          }
        }
        ot[ml * RS + nl] = OUT_DT == IC_DTYPE_F16 ? f32_to_f16(v) : f32_to_bf16(v);
      }
  }
  __syncthreads();
  for (int c = tid; c < BM * CPR; c += kMT) {
    const int row = c / CPR, col = (c % CPR) * 8, m = m0 + row, n = n0 + col;
    if (m < M && n < N) *(v4u*)((u16*)C + (int64_t)m * ldc + n) = *(const v4u*)(ot + row * RS + col);
  }
}

// Ring depths that let two (packed 32- and 64-row tiles: three or four)
// workgroups share a CU's 160 KB of LDS.
template <int T, int MODE>
using MidCfg = mid::Cfg<kMidTile[T].bm / 32, kMidTile[T].bn / 32,
                        T < 2 ? 4 : (T == 3 && MODE == big::ROW8 ? 2 : 3), MODE>;

template <int T, int MODE, int OUT_DT, bool EPI, bool KIL, bool PART>
hipError_t launch_mid_k(const ic_gemm::GemmArgs& g, int S, hipStream_t st) {
  using CF = MidCfg<T, MODE>;
  // LDS goes in 512-byte granules; the registers (at most 116) hold as many workgroups
  static_assert(kMidCost[MODE].wgs[T] == 163840 / ((CF::lds_bytes + 511) / 512 * 512),
                "the plan's workgroups per CU");
  const int tiles = ((g.M + CF::BM - 1) / CF::BM) * ((g.N + CF::BN - 1) / CF::BN);
  auto kern = gemm_mid_kernel<CF, OUT_DT, EPI, KIL, PART>;
  static unsigned char lds_set[64];  // per device
  if (hipError_t e = ic_set_lds_limit((const void*)kern, (int)CF::lds_bytes, lds_set)) return e;
  kern<<<dim3(tiles, S), dim3(mid::kMT), CF::lds_bytes, st>>>(g.A, g.lda, g.B, g.ldb, g.s_a, g.s_w, g.G, g.bias,
                                                              g.bias_dt, g.C, g.ldc, g.M, g.N, g.K, (int32_t*)g.ws,
                                                              g.epi);
  return hipGetLastError();
}

// One launch (S = 1), or S slices and their reduction (g.ws holds
// 4 * S * M * N bytes).  W16: A rows in bytes, no EPI.
template <int T, int MODE, bool KIL, int OUT_DT>
hipError_t launch_mid_t(const ic_gemm::GemmArgs& g, int S, hipStream_t st) {
  const bool epi = g.epi.act != 0 || g.epi.res != nullptr;
  if (S == 1) {
    if constexpr (MODE != big::W16) {
      if (epi) return launch_mid_k<T, MODE, OUT_DT, true, KIL, false>(g, 1, st);
    }
    return launch_mid_k<T, MODE, OUT_DT, false, KIL, false>(g, 1, st);
  }
  // the partials do not depend on the output type, except through W4A16's dequantization
  constexpr int PDT = MODE == big::W16 ? OUT_DT : IC_DTYPE_BF16;
  if (hipError_t e = launch_mid_k<T, MODE, PDT, false, KIL, true>(g, S, st)) return e;
  constexpr int KIND = MODE == big::ROW8 ? 0 : (MODE == big::ROW4 ? 1 : (MODE == big::W16 ? 3 : 2));
  const int64_t q = (int64_t)g.M * g.N / 4;
  splitk_reduce4_kernel<KIND, OUT_DT><<<dim3((unsigned)((q + 255) / 256)), dim3(256), 0, st>>>(
      (const int32_t*)g.ws, S, g.s_a, g.s_w, g.bias, g.bias_dt, g.C, g.ldc, g.M, g.N, g.epi);
  return hipGetLastError();
}
template <int MODE, bool KIL, int OUT_DT>
hipError_t launch_mid_d(const ic_gemm::GemmArgs& g, int tile, int S, hipStream_t st) {
  switch (tile) {
    case 0: return launch_mid_t<0, MODE, KIL, OUT_DT>(g, S, st);
    case 1: return launch_mid_t<1, MODE, KIL, OUT_DT>(g, S, st);
    case 2:
      if constexpr (MODE != big::ROW4) return launch_mid_t<2, MODE, KIL, OUT_DT>(g, S, st);
      break;
    case 3:
      if constexpr (MODE == big::ROW8 || MODE == big::W16) return launch_mid_t<3, MODE, KIL, OUT_DT>(g, S, st);
  }
  return hipErrorInvalidValue;
}
template <int MODE, bool KIL>
hipError_t launch_mid(const ic_gemm::GemmArgs& g, int tile, int S, hipStream_t st) {
  if (g.out_dt == IC_DTYPE_F16) return launch_mid_d<MODE, KIL, IC_DTYPE_F16>(g, tile, S, st);
  return launch_mid_d<MODE, KIL, IC_DTYPE_BF16>(g, tile, S, st);
}

}  // namespace
