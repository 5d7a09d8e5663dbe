// Rows, waves and row scales of the FP32 MTE workgroups (host code without HIP,
// so that a host program can run it).
#ifndef ROADMC_MTE_PLAN_H
#define ROADMC_MTE_PLAN_H

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "roadmc.h"

namespace roadmc {

constexpr int kMteGranule = 32;           // rows and columns of an output tile
constexpr int kMteTilesFourWaves = 16;    // output tiles that four waves hold
constexpr size_t kMteLdsPerCu = 160 * 1024;

// One (road, species) job: padded patches, paths, and the rows of its bucket's
// tile setting (capped by the paths and the tile budget).
struct MtePlanJob {
  int Pp;
  int64_t N;
  int rows;
};
struct MtePlanTile {
  int rows, waves;
};

// Rows: the tile table's, halved (down to 32) while the launch has fewer
// workgroups than the card has CUs, since a path's result does not depend on
// them: 256 patches and 5,000 paths 1.27 -> 0.84 ms, 100 patches and 2,000
// paths 0.78 -> 0.54 ms.
// Waves: tiles of at most 16 output tiles run as four-wave workgroups, two of
// them on a CU (see mte_kernels.hip); larger ones, those whose LDS leaves no
// room for a second and those of a launch without a second workgroup for some
// CU as eight-wave workgroups.
// nominal (the tuner): the rows of the tile table whatever the launch's size
// and the waves of a launch that fills the card, so that a setting is timed in
// the form it is kept for.  With 2,048 paths the halving ran the trials of 64,
// 128 and 256 rows as one and the same launch, and noise chose between them.
// lds(rows, Pp): the workgroup's dynamic LDS.
template <class Lds>
std::vector<MtePlanTile> mte_plan_f32(const std::vector<MtePlanJob>& jobs, int n_cu, bool nominal,
                                      const Lds& lds) {
  int shrink = 1;
  auto rows_of = [&](const MtePlanJob& j) {
    return std::max(kMteGranule, j.rows / shrink / kMteGranule * kMteGranule);
  };
  auto workgroups = [&]() {
    int64_t n = 0;
    for (const MtePlanJob& j : jobs) n += (j.N + rows_of(j) - 1) / rows_of(j);
    return n;
  };
  while (!nominal && shrink < 8 && workgroups() < n_cu) shrink *= 2;
  const bool fills = nominal || workgroups() > n_cu;
  std::vector<MtePlanTile> out;
  out.reserve(jobs.size());
  for (const MtePlanJob& j : jobs) {
    const int rows = rows_of(j), ntiles = rows / kMteGranule * (j.Pp / kMteGranule);
    const bool four = fills && ntiles <= kMteTilesFourWaves && 2 * lds(rows, j.Pp) <= kMteLdsPerCu;
    out.push_back({rows, four ? 4 : 8});
  }
  return out;
}

// Whether the paths of a job differ, but by little: a year's noise of a
// population between 0 and 5e-3 of it (at a fifth of the capacity from the
// capacity, for the laws whose noise is in the growth rate).  The FP32 kernels
// then scale the rows (TraitsX6): a patch's mean over 4,000 paths of 1,000
// patches is 9.1e-8 off unscaled against 6.7e-8 scaled at a noise of 1e-3, and
// 4.2e-8 either way at 1e-2.  Not without noise: equal paths round alike on any
// unit, and unscaled an exact product stays exact (populations that nothing
// changes keep their total, and meet a threshold of all of it).
inline bool mte_low_noise(int law, double dt, double noise_sd, const double params[8]) {
  double e = std::fabs(noise_sd);
  if (law == ROADMC_LAW_REF_CPU) e = 0.2 * std::fabs(dt * params[2]) * 0.01;
  if (law == ROADMC_LAW_REF_GPU)
    e = 0.2 * std::max(std::fabs(params[0]), std::fabs(params[1])) *
        std::max({std::fabs(params[2]), std::fabs(params[7]),
                  params[6] > 0.0 ? std::fabs(params[5]) : 0.0});
  return e > 0.0 && e < 5e-3;
}

}  // namespace roadmc

#endif
