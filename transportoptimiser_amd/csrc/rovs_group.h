// Plan, LDS layout and row grouping of the policy kernels (rovs_kernels.hip):
// the parts that decide which LDS word is written, apart from the device
// intrinsics, so that a host program can run them over every plan.  Compiles
// as C++ (host tools) and as HIP.
#ifndef ROADMC_ROVS_GROUP_H
#define ROADMC_ROVS_GROUP_H

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "rng.h"  // RMC_HD

namespace roadmc {

constexpr int kRgWaves = 8, kRgThreads = kRgWaves * 64;
constexpr int kRgTiles = 12;  // group tiles of the row map: 160 rows of 8 controls
constexpr int kRgMaxRows = 160;
constexpr int kRgParts = 4;  // column quarters of a row's dots
constexpr int kRgPad = 4;    // floats between the tile's rows (TraitsX6::PAD)
constexpr size_t kRgLdsMax = 160 * 1024;

// Column tiles a wave owns, and the group tiles whose products it can hold:
// 7 (an eighth spills in the product loop) or 4 of two columns.
inline int rg_cols(int Pp) { return Pp > 32 * kRgWaves ? 2 : 1; }
#if defined(__HIPCC__)
__host__ __device__
#endif
constexpr int rg_slots(int cols) { return cols == 1 ? 7 : 4; }

// Group tiles that BM rows under C controls can need, and those that a
// workgroup's waves can hold: up to 128 patches two or four waves share a
// column tile and split the group tiles between them.  Without that eight
// controls took the dense form there, whose products two (64 patches) or four
// of the eight waves form: at 64 patches, 20,000 paths, 10 years 433 us forward
// and 706 us reverse against 122 and 186 us grouped.
inline int rg_max_tiles(int BM, int C) { return (BM - std::min(C, BM)) / 32 + std::min(C, BM); }
inline int rg_capacity(int Pp) {
  const int ntc = Pp / 32;
  return std::min(kRgTiles, rg_slots(rg_cols(Pp)) * (ntc <= kRgWaves ? kRgWaves / ntc : 1));
}

struct RgPlan {
  int BM;
  int dense;  // 32 rows, every used control's product, selected per path
  size_t lds;
};

// LDS: n_tiles tiles, then [kRgParts][C + 1][BM] partial dots, [n_st][C + 1][BM]
// dots, growth-rate means, totals or coefficients, controls, the row map
// ([kRgTiles][32]) and the tiles' controls.
inline size_t rg_lds(int BM, int Pp, int C, int n_tiles, int n_st) {
  return sizeof(float) * ((size_t)n_tiles * BM * (Pp + kRgPad) +
                          (size_t)(kRgParts + n_st) * (C + 1) * BM + 3 * (size_t)BM +
                          kRgTiles * 32 + 16);
}

// The rows of a launch over N paths: of the sizes (whole path quads) that LDS
// and the waves' registers allow, the one with the least rounds of workgroups
// over the n_cu CUs times work, in product tiles: 1.6 for 32 paths (product, growth
// and dots) and half a tile of padding per control.  The results do not depend
// on the rows.
inline RgPlan rg_plan(int N, int Pp, int C, int n_tiles, int n_st, int n_cu) {
  RgPlan best{32, 0, rg_lds(32, Pp, C, n_tiles, n_st)};
  best.dense = rg_max_tiles(8, C) > rg_capacity(Pp);
  double cost = 1e300;
  for (int BM = 8; BM <= kRgMaxRows; BM += 4) {
    const size_t lds = rg_lds(BM, Pp, C, n_tiles, n_st);
    if (lds > kRgLdsMax || rg_max_tiles(BM, C) > rg_capacity(Pp)) continue;
    const int rounds = ((N + BM - 1) / BM + n_cu - 1) / n_cu;
    const double c = rounds * (1.6 * BM / 32 + 0.5 * C);
    if (c < cost) {
      cost = c;
      best = RgPlan{BM, 0, lds};
    }
  }
  return best;
}

struct RgShape {
  int BM, Pp, LDA, nch, C, dense;
};

// LDS arrays after the tiles.
struct RgArrays {
  float *part, *st, *grm, *aux;
  int *ctl, *map, *tiles;
};
RMC_HD RgArrays rg_arrays(const RgShape& sh, float* smem, int n_tiles, int n_st) {
  RgArrays r;
  r.part = smem + (size_t)n_tiles * sh.BM * sh.LDA;
  r.st = r.part + kRgParts * (sh.C + 1) * sh.BM;
  r.grm = r.st + n_st * (sh.C + 1) * sh.BM;
  r.aux = r.grm + sh.BM;
  r.ctl = reinterpret_cast<int*>(r.aux + sh.BM);
  r.map = r.ctl + sh.BM;
  r.tiles = r.map + kRgTiles * 32;
  return r;
}

// One wave, rg_group_clear in every lane before rg_group_fill in any: map
// [tile][32] holds the row of each group slot (-1 in the padding), tiles[t] the
// control of group tile t and tiles[kRgTiles] their number.  ctl is -1 for rows
// past the last path.  ballot(i, v, c) is the mask of the lanes whose v, the
// control of row 64 i + lane, is c.
// The dense form has no groups (its controls can make more than kRgTiles) and
// writes nothing here.
RMC_HD void rg_group_clear(const RgShape& sh, int* map, int lane) {
  if (sh.dense) return;
#pragma GCC unroll 4
  for (int i = 0; i < kRgTiles * 32; i += 64)
    if (i + lane < kRgTiles * 32) map[i + lane] = -1;
}
template <class Ballot>
RMC_HD void rg_group_fill(const RgShape& sh, const int* ctl, int* map, int* tiles, int lane,
                          const Ballot& ballot) {
  if (sh.dense) return;
  const int c0 = lane < sh.BM ? ctl[lane] : -1;
  const int c1 = 64 + lane < sh.BM ? ctl[64 + lane] : -1;
  const int c2 = 128 + lane < sh.BM ? ctl[128 + lane] : -1;
  auto count = [](uint64_t m) { return __builtin_popcountll(m); };
  const uint64_t below = (1ull << lane) - 1;
  int nt = 0;
  for (int c = 0; c < sh.C; ++c) {
    const uint64_t m0 = ballot(0, c0, c), m1 = ballot(1, c1, c), m2 = ballot(2, c2, c);
    const int n0 = count(m0), n1 = n0 + count(m1), n = n1 + count(m2);
    if (c0 == c) map[32 * nt + count(m0 & below)] = lane;
    if (c1 == c) map[32 * nt + n0 + count(m1 & below)] = 64 + lane;
    if (c2 == c) map[32 * nt + n1 + count(m2 & below)] = 128 + lane;
    const int k = (n + 31) >> 5;
    if (lane < k) tiles[nt + lane] = c;
    nt += k;
  }
  if (lane == 0) tiles[kRgTiles] = nt;
}

}  // namespace roadmc

#endif
