// Choice of the small-tile kernel (gemm_mid.h) and its K split: host logic
// shared by the INT8 and W4A16 entry points.
//
// Estimated microseconds, fitted to launches timed on MI355X (bf16 outputs, back
// to back in a graph, weights cycling through three copies; 746 shapes and more of
// 17 to 3072 rows, 64 to 18432 columns and K 128 to 14336 per mode, each tile and slice
// count by itself: 5 to 8 % rms).  A CU takes its workgroups in turns of
// as many as its LDS holds (`wgs`); in a turn of n a stage takes max(lat, n *
// thr), and a turn ends with `end` (its epilogue).  Where a tile's stage is
// bound by the VALU's folds (groups of 64 and 32 columns) the turns do not show
// and wgs is 0, any number at once.
//   W4A16  512 x 9216 x 3072: 128 x 64 tiles, three per CU in two turns, 81 us;
//          256 x 192 tiles 65 (128 x 128: 71)
//   W4A16  768 x 18432 x 3072: 128 x 128 139; 256 x 256 tiles in one turn 90
//   W8A8   2048 x 12288 x 3072: 128 x 128 82; 256 x 192 72.6; 512 x 3072 x 3072:
//          64 x 64 tiles 12.8, 256 x 192 in two slices 25.4
//   g128   640 x 12288 x 3072: 128 x 64 48; 256 x 192 43
//   int8 weights in groups, 384 x 18432 x 3072: 64 x 64 54; 256 x 192 43.4
//   g64    146 x 1312 x 8448: 32 x 64 29.7, 64 x 64 43.1; 256 x 192 125.5
// Past two rounds of the large tiles the small ones are not looked at
// (mid_rounds_ok).
#pragma once
#include "gemm_common.h"

namespace {

struct MidTile { int bm, bn; };
constexpr int kMidTiles = 4;
constexpr MidTile kMidTile[kMidTiles] = {{32, 64}, {64, 64}, {128, 64}, {128, 128}};

struct MidCost {
  double fixed, reduce, bytes;  // of a launch; a split's second kernel, and its partials (8 bytes each) per us
  int wgs[kMidTiles];
  double lat[kMidTiles], thr[kMidTiles], end[kMidTiles];  // lat 0: the mode has no such tile
};
// by weight mode (big::G128 ... big::W16): 128-K stages, 64-K for W16
constexpr MidCost kMidCost[7] = {
    {5.66, 2.35, 3.47e6, {4, 3, 2, 0},
     {0.22, 0.42, 0.64, 0}, {0.195, 0.243, 0.405, 0}, {0.27, 0.56, 0.98, 0}},  // G128
    {3.0, 2.5, 5.0e6, {0, 0, 0, 0}, {0.39, 0.60, 0.80, 0}, {0.22, 0.33, 0.55, 0}, {0, 0, 0, 0}},  // G64
    {5.37, 1.87, 3.42e6, {5, 3, 2, 0},
     {0.21, 0.35, 0.47, 0}, {0.140, 0.186, 0.325, 0}, {0.41, 0.44, 0.54, 0}},  // ROW4
    {5.57, 3.03, 3.88e6, {3, 2, 2, 2},
     {0.20, 0.26, 0.45, 0.74}, {0.204, 0.200, 0.309, 0.428}, {0.26, 0.91, 0.86, 1.20}},  // ROW8
    {3.0, 2.5, 5.0e6, {0, 0, 0, 0}, {0.62, 0.95, 1.40, 0}, {0.40, 0.60, 1.05, 0}, {0, 0, 0, 0}},  // G32
    {5.39, 3.41, 5.12e6, {3, 2, 2, 0},
     {0.23, 0.35, 0.54, 0}, {0.193, 0.258, 0.407, 0}, {0.38, 1.36, 1.33, 0}},  // G128I8
    {5.82, 2.96, 5.62e6, {6, 3, 2, 2},
     {0.43, 0.44, 0.60, 0.90}, {0.294, 0.303, 0.414, 0.711}, {0.02, 0, 0.44, 0.13}},  // W16
};
// The launches the small tiles stand in for: the big tiles (a stage of 256 rows;
// W16 on 192 columns) and the tile kernel (a 128 x 128 stage and each further
// 128 x 128 of a larger tile, per turn one workgroup of a CU).
struct LargeCost { double fixed, stage, end, t_fixed, one, more, t_end, reduce, bytes; };
constexpr LargeCost kLargeCost[7] = {
    {3.64, 1.26, 6.72, 3.64, 0.82, 0.37, 3.28, 2.55, 4.14e6},  // G128
    {5.0, 1.8, 4.0, 0, 0, 0, 0, 0, 1},                         // G64
    {4.90, 0.91, 7.52, 4.88, 0.72, 0.26, 1.84, 1.81, 2.99e6},  // ROW4
    {2.17, 1.08, 5.07, 4.88, 0.48, 0.34, 2.19, 6.34, 3.94e6},  // ROW8
    {5.0, 3.5, 4.0, 0, 0, 0, 0, 0, 1},                         // G32
    {2.34, 1.49, 7.94, 2.34, 0.64, 0.40, 3.74, 3.28, 4.31e6},  // G128I8
    {6.92, 1.24, 0.0, 0, 0, 0, 0, 0, 1},                       // W16
};

bool mid_rounds_ok(int64_t M, int64_t N) {
  return ((M + 255) / 256) * ((N + 191) / 192) <= 2 * (int64_t)ic_num_cus();
}

struct MidPlan { int tile, S; double us; };
// KT: K stages of the mode; between min_s and max_s slices (of at least four
// stages each, unless min_s asks for them)
MidPlan mid_plan(int mode, int64_t M, int64_t N, int KT, int min_s, int max_s) {
  const int64_t cus = ic_num_cus();
  MidPlan best{0, 1, 1e30};
  const MidCost& c = kMidCost[mode];
  for (int t = 0; t < kMidTiles; ++t) {
    if (c.lat[t] == 0) continue;
    const auto stage = [&](int64_t n) { return n * c.thr[t] > c.lat[t] ? n * c.thr[t] : c.lat[t]; };
    const int64_t tiles = ((M + kMidTile[t].bm - 1) / kMidTile[t].bm) * ((N + kMidTile[t].bn - 1) / kMidTile[t].bn);
    for (int S = min_s; S <= max_s && (S == min_s || KT / S >= 4); ++S) {
      const int64_t load = (tiles * S + cus - 1) / cus, wgs = c.wgs[t] > 0 ? c.wgs[t] : load;
      const int64_t turns = (load + wgs - 1) / wgs, rest = load % wgs;
      const double per = (load / wgs) * stage(wgs) + (rest > 0 ? stage(rest) : 0.0);
      const double us = c.fixed + (KT + S - 1) / S * per + turns * c.end[t] +
                        (S > 1 ? c.reduce + (double)S * M * N * 8.0 / c.bytes : 0.0);
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
