/* The policy kernels' plan and row grouping (rovs_group.h), run on the host one
 * wave at a time over every plan that a valuation's sizes can reach: the
 * grouping stays inside its LDS arrays, puts each path into one slot of its own
 * control in path order, and takes no more tiles than the waves hold. */
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "rovs_group.h"

using namespace roadmc;

static int failures = 0;
#define CHECK(x)                                                                                \
  do {                                                                                          \
    if (!(x) && ++failures <= 20)                                                               \
      printf("C=%d Pp=%d rows=%d dense=%d pattern=%d: %s\n", sh.C, sh.Pp, sh.BM, sh.dense,       \
             pattern, #x);                                                                      \
  } while (0)

static void group(const RgShape& sh, size_t lds, int n_tiles, int rows, int pattern) {
  constexpr int kGuard = 64, kMark = 0x5aa5c33c;
  const size_t words = lds / 4;
  std::vector<int> mem(words + kGuard, kMark);
  const RgArrays L = rg_arrays(sh, reinterpret_cast<float*>(mem.data()), n_tiles, 1);
  CHECK(L.tiles + kRgTiles < mem.data() + words);
  unsigned x = 12345u + 977u * pattern + sh.C;
  for (int r = 0; r < sh.BM; ++r) {
    x = x * 1664525u + 1013904223u;
    const int c = pattern == 0   ? (int)((x >> 16) % sh.C)        // random
                  : pattern == 1 ? (r < sh.C ? r : sh.C - 1)      // one each, the rest the last
                  : pattern == 2 ? (r < sh.C ? r : 0)             // the rest the first
                                 : sh.C - 1;                      // one control
    L.ctl[r] = r < rows ? c : -1;
  }
  auto mask = [&](int i, int, int c) -> uint64_t {
    uint64_t m = 0;
    for (int l = 0; l < 64; ++l)
      if (64 * i + l < sh.BM && L.ctl[64 * i + l] == c) m |= 1ull << l;
    return m;
  };
  // Words past the arrays of the grouping may not change; the vector's tail
  // takes the writes that would leave the workgroup's LDS.
  for (int l = 0; l < 64; ++l) rg_group_clear(sh, L.map, l);
  for (int l = 0; l < 64; ++l) rg_group_fill(sh, L.ctl, L.map, L.tiles, l, mask);
  for (int i = kRgTiles + 1; L.tiles + i < mem.data() + mem.size(); ++i)
    CHECK(L.tiles[i] == kMark);
  if (sh.dense) {
    // No reader of the map or the tiles in this form: nothing is written.
    for (int i = 0; i < kRgTiles * 32 + kRgTiles + 1; ++i) CHECK(L.map[i] == kMark);
    return;
  }
  const int nt = L.tiles[kRgTiles];
  // rg_move: the waves that share a column tile split the group tiles evenly.
  const int ntc = sh.Pp / 32, share = ntc <= kRgWaves ? kRgWaves / ntc : 1;
  CHECK(nt >= 0 && nt <= kRgTiles && (nt + share - 1) / share <= rg_slots(rg_cols(sh.Pp)));
  std::vector<int> seen(sh.BM, 0);
  int last_c = -1, last_r = -1;
  for (int s = 0; s < kRgTiles * 32; ++s) {
    const int r = L.map[s];
    if (r < 0) continue;
    CHECK(s < 32 * nt && r < rows && r < sh.BM);
    if (s >= 32 * nt || r >= sh.BM) return;
    CHECK(L.ctl[r] == L.tiles[s / 32]);
    CHECK(L.ctl[r] > last_c || (L.ctl[r] == last_c && r > last_r));
    last_c = L.ctl[r];
    last_r = r;
    ++seen[r];
  }
  for (int r = 0; r < sh.BM; ++r) CHECK(seen[r] == (r < rows ? 1 : 0));
}

int main() {
  int rows_seen[3] = {0, 0, 0}, dense_seen = 0;
  for (int C = 1; C <= 8; ++C)
    for (int Pp = 64; Pp <= 512; Pp += 64)
      for (int n_tiles = 1; n_tiles <= 2; ++n_tiles)
        for (int N : {1, 7, 40, 300, 5000, 9000, 20000, 30000, 100000, 1000000}) {
          const RgPlan pl = rg_plan(N, Pp, C, n_tiles, 1, 256);
          const RgShape sh{pl.BM, Pp, Pp + kRgPad, Pp / 16, C, pl.dense};
          const int pattern = -1;
          CHECK(pl.BM >= 8 && pl.BM <= kRgMaxRows && pl.BM % 4 == 0);
          CHECK(pl.lds == rg_lds(pl.BM, Pp, C, n_tiles, 1) && pl.lds <= kRgLdsMax);
          CHECK(!pl.dense || pl.BM == 32);
          // Every control's product only where the waves cannot hold the
          // groups: never where two or more waves share a column tile.
          CHECK(pl.dense == ((C == 8 && Pp > 128) || (C > 4 && Pp > 256)));
          rows_seen[pl.BM > 128 ? 2 : pl.BM > 64 ? 1 : 0] = 1;
          dense_seen |= pl.dense;
          // The plan follows the device: half the CUs take half the paths in
          // the same rounds.
          CHECK(rg_plan(N, Pp, C, n_tiles, 1, 128).BM == rg_plan(2 * N, Pp, C, n_tiles, 1, 256).BM);
          for (int p = 0; p < 4; ++p)
            for (int rows : {pl.BM, pl.BM - 3, 1}) group(sh, pl.lds, n_tiles, rows, p);
        }
  // The rows that the GPU test's sizes are meant to reach.
  const int reach[][5] = {{33001, 64, 3, 132, 132}, {39985, 64, 8, 160, 160},
                          {20005, 128, 7, 80, 80},  {30011, 192, 3, 120, 60},
                          {33003, 256, 2, 132, 68}, {10011, 320, 2, 40, 40}};
  for (const auto& r : reach)
    for (int n_tiles = 1; n_tiles <= 2; ++n_tiles) {
      const RgPlan pl = rg_plan(r[0], r[1], r[2], n_tiles, 1, 256);
      const RgShape sh{pl.BM, r[1], r[1] + kRgPad, r[1] / 16, r[2], pl.dense};
      const int pattern = -1;
      CHECK(pl.BM == r[2 + n_tiles] && !pl.dense);
    }
  printf("%s: rows up to 64 %d, 128 %d, 160 %d, dense %d, failures %d\n",
         failures ? "FAILED" : "ok", rows_seen[0], rows_seen[1], rows_seen[2], dense_seen,
         failures);
  return failures ? 1 : 0;
}
