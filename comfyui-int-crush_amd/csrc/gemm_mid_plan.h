// Choice of the small-tile kernel (gemm_mid.h) and its K split: host logic
// shared by the INT8 and W4A16 entry points.
//
// Times in microseconds, from launches measured on MI355X (bf16 outputs,
// weights cycling through three copies).  A tile's stage takes `lat` alone on
// its CU and `thr` for each workgroup that shares it:
//   W8A8   512 x 3072 x 3072 (24 stages): 64 x 64 tiles, 384 of them, 12.8 us;
//          32 x 64 14.4, 128 x 64 15.5, 128 x 128 19.5; 256 x 192 in two
//          slices 25.4
//   W8A8   77 x 4096 x 4096: 32 x 64 9.2, 64 x 64 11.4; 128 x 128 in eight
//          slices 16.5
//   g64    146 x 1312 x 8448: 32 x 64 29.7, 64 x 64 43.1; 256 x 192 125.5
//   W4A16  63 x 3256 x 3712: 64 x 64 33.8, in four slices 16.5; 128 x 256 68.9
// The large tiles stay ahead once they fill the CUs (W8A8 1111 x 9216 x 3072:
// 35.6 against 43.8 us; g128 1357 x 7688 x 2560: 40.7 against 49.4), and past
// two rounds of them the small ones are not looked at (mid_rounds_ok): the
// estimates leave out the epilogues' memory time, which weighs on short K
// (W8A8 19053 x 10992 x 1152 with GELU and a residual: 608 us on 320 x 192
// tiles, 624 us on 128 x 128).
#pragma once
#include "gemm_common.h"

namespace {

struct MidTile { int bm, bn; };
constexpr int kMidTiles = 4;
constexpr MidTile kMidTile[kMidTiles] = {{32, 64}, {64, 64}, {128, 64}, {128, 128}};

struct MidCost { double lat[kMidTiles], thr[kMidTiles]; };  // 0: the mode has no such tile
// by weight mode (big::G128 ... big::W16): 128-K stages, 64-K for W16
constexpr MidCost kMidCost[7] = {
    {{0.27, 0.36, 0.55, 0}, {0.175, 0.28, 0.42, 0}},        // G128
    {{0.39, 0.60, 0.80, 0}, {0.22, 0.33, 0.55, 0}},         // G64
    {{0.25, 0.32, 0.52, 0}, {0.17, 0.25, 0.38, 0}},         // ROW4
    {{0.21, 0.265, 0.48, 0.61}, {0.16, 0.21, 0.36, 0.42}},  // ROW8
    {{0.62, 0.95, 1.40, 0}, {0.40, 0.60, 1.05, 0}},         // G32
    {{0.30, 0.42, 0.57, 0}, {0.21, 0.26, 0.46, 0}},         // G128I8
    {{0.48, 0.54, 0.75, 0.98}, {0.27, 0.32, 0.43, 0.65}},   // W16
};
// fixed part of a launch; the second kernel of a split and its partials' round trip
constexpr double kMidFixed = 3.0, kMidReduce = 2.5, kMidBytesPerUs = 5e6;

bool mid_rounds_ok(int64_t M, int64_t N) {
  return ((M + 255) / 256) * ((N + 191) / 192) <= 2 * (int64_t)ic_num_cus();
}

struct MidPlan { int tile, S; double us; };
// KT: K stages of the mode; between min_s and max_s slices (of at least four
// stages each, unless min_s asks for them)
MidPlan mid_plan(int mode, int64_t M, int64_t N, int KT, int min_s, int max_s) {
  const int64_t cus = ic_num_cus();
  MidPlan best{0, 1, 1e30};
  for (int t = 0; t < kMidTiles; ++t) {
    const double lat = kMidCost[mode].lat[t], thr = kMidCost[mode].thr[t];
    if (lat == 0) continue;
    const int64_t tiles = ((M + kMidTile[t].bm - 1) / kMidTile[t].bm) * ((N + kMidTile[t].bn - 1) / kMidTile[t].bn);
    for (int S = min_s; S <= max_s && (S == min_s || KT / S >= 4); ++S) {
      int64_t load = (tiles * S + cus - 1) / cus;
      if (t == 3 && load > 1) load = (load + 1) & ~1;  // two at a time: an odd one leaves half its CU idle
      const double per = load * thr > lat ? load * thr : lat;
      const double us = kMidFixed + (KT + S - 1) / S * per +
                        (S > 1 ? kMidReduce + (double)S * M * N * 8.0 / kMidBytesPerUs : 0.0);
      if (us < best.us) best = {t, S, us};
    }
  }
  return best;
}

}  // namespace

// One launch of gemm_mid_kernel on tile `tile` (S = 1), or S K slices into g.ws
// and their reduction.  g: 16-bit, 16-byte aligned output (and residual) with
// row strides and N multiples of 8; W16: A rows in bytes, g.kil the staged
// layout, no activation or residual.
hipError_t ic_launch_mid_i4(const ic_gemm::GemmArgs& g, int mode, int tile, int S, hipStream_t st);
hipError_t ic_launch_mid_kil(const ic_gemm::GemmArgs& g, int mode, int tile, int S, hipStream_t st);
hipError_t ic_launch_mid_i8(const ic_gemm::GemmArgs& g, int mode, int tile, int S, hipStream_t st);
hipError_t ic_launch_mid_w16(const ic_gemm::GemmArgs& g, int tile, int S, hipStream_t st);
// ic_gemm_route for W4A16 (gemm_w4a16.hip)
void ic_w4a16_route(int64_t M, int64_t N, int64_t K, int64_t num_groups, int64_t ws_bytes, int32_t* route);
