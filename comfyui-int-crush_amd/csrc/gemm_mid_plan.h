// Choice of the small-tile kernel (gemm_mid.h) and its K split: host logic
// shared by the INT8 and W4A16 entry points.
//
// Estimated microseconds, their constants set so that the choice they lead to is
// right on launches timed on MI355X (bf16 outputs, back to back in a graph, weights
// cycling through three copies; 1700 shapes per mode, W4A16 746, of 17 to 4608
// rows, 64 to 18432 columns and K 128 to 14336, each tile by itself: of 11914
// launches 12 were more than 4 % slower than the large tiles, by at most 9 %, and 59
// more than 6 % slower than the best tile).  A CU takes its workgroups in turns of
// as many as its LDS holds (`wgs`); in a turn of n a stage takes max(lat, n *
// thr), and a turn ends with `end` (its epilogue).
//   W4A16  512 x 9216 x 3072: 128 x 64 tiles, three per CU in two turns, 81 us;
//          256 x 192 tiles 65 (128 x 128: 71)
//   W4A16  768 x 18432 x 3072: 128 x 128 139; 256 x 256 tiles in one turn 90
//   per-row INT4, 4608 x 5120 x 512: 128 x 64 tiles in six turns, whose ends weigh
//          at short K, 34.6; 256 x 192 25.1
//   g64    513 x 18432 x 512: 128 x 64 24; 256 x 192 18.1
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
  int wgs[kMidTiles];  // workgroups that a CU's LDS holds
  double lat[kMidTiles], thr[kMidTiles], end[kMidTiles];  // lat 0: the mode has no such tile
};
// by weight mode (big::G128 ... big::W16): 128-K stages, 64-K for W16
constexpr MidCost kMidCost[7] = {
    {3.45, 2.81, 3.63e6, {4, 3, 2, 0},
     {0.219, 0.407, 0.728, 0}, {0.205, 0.272, 0.41, 0}, {0.873, 0.973, 1.813, 0}},  // G128
    {1.98, 5.69, 11.45e6, {4, 3, 2, 0},
     {0.506, 0.58, 0.82, 0}, {0.241, 0.361, 0.642, 0}, {1.729, 1.736, 1.797, 0}},  // G64
    {6.12, 1.87, 3.42e6, {5, 3, 0, 0},
     {0.21, 0.35, 0, 0}, {0.140, 0.186, 0, 0}, {0.605, 0.61, 0, 0}},  // ROW4 (128 x 64 led at 8 of 1718 shapes, by 3 to 5 %: left out)
    {4.88, 3.03, 3.88e6, {3, 2, 2, 2},
     {0.20, 0.26, 0.45, 0.74}, {0.204, 0.200, 0.309, 0.428}, {0.279, 1.206, 1.694, 2.295}},  // ROW8
    {3.05, 1.65, 3.39e6, {4, 3, 2, 0},
     {0.704, 0.702, 1.298, 0}, {0.349, 0.557, 1.183, 0}, {1.458, 1.72, 2.974, 0}},  // G32
    {4.73, 3.64, 6.08e6, {3, 2, 2, 0},
     {0.299, 0.548, 0.599, 0}, {0.193, 0.268, 0.382, 0}, {0.516, 1.208, 1.409, 0}},  // G128I8
    {5.82, 2.96, 5.62e6, {6, 3, 2, 2},
     {0.43, 0.44, 0.60, 0.90}, {0.294, 0.303, 0.414, 0.711}, {0.02, 0, 0.44, 0.13}},  // W16
};
// The launches the small tiles stand in for: the big tiles (a stage of 256 rows;
// W16 on 192 columns) and the tile kernel (a 128 x 128 stage and each further
// 128 x 128 of a larger tile, per turn one workgroup of a CU).
struct LargeCost { double fixed, stage, end, t_fixed, one, more, t_end, reduce, bytes; };
constexpr LargeCost kLargeCost[7] = {
    {1.821, 1.651, 4.001, 2.496, 0.843, 0.396, 3.354, 4.245, 4.762e6},  // G128
    {0.18, 2.34, 4.939, 0, 0, 0, 0, 0, 1},  // G64
    {2.19, 1.198, 5.191, 6.188, 0.695, 0.216, 1.296, 3.453, 4.185e6},  // ROW4
    {4.005, 1.094, 4.838, 4.318, 0.382, 0.394, 2.022, 5.927, 4.962e6},  // ROW8
    {0.136, 4.487, 7.407, 0, 0, 0, 0, 0, 1},  // G32
    {3.027, 1.518, 4.94, 2.34, 0.546, 0.533, 3.74, 3.28, 4.965e6},  // G128I8
    {6.92, 1.24, 0.0, 0, 0, 0, 0, 0, 1},  // W16
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
      const int64_t load = (tiles * S + cus - 1) / cus, wgs = c.wgs[t];
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
