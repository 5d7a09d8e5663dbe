/* The FP32 MTE launch plan (mte_plan.h) on the host. */
#include <cstdio>

#include "mte_plan.h"

using namespace roadmc;

static int failures = 0;
#define CHECK(x)                                       \
  do {                                                 \
    if (!(x)) {                                        \
      ++failures;                                      \
      printf("line %d: %s\n", __LINE__, #x);           \
    }                                                  \
  } while (0)

static size_t lds(int rows, int Pp) { return (size_t)rows * (Pp + 5) * 4 + 256; }

int main() {
  // The tuner's eight roads: a trial runs the rows it is kept for, in the form
  // of a launch that fills the card, however few its paths.
  for (int64_t N : {256, 2048, 20000, 1000000})
    for (int Pp : {96, 128, 256, 512, 1024})
      for (int rows = 32; rows <= 256 && rows * Pp <= 32768; rows *= 2) {
        const std::vector<MtePlanJob> jobs(8, MtePlanJob{Pp, N, rows});
        const auto full = mte_plan_f32(std::vector<MtePlanJob>(8, MtePlanJob{Pp, 1 << 20, rows}),
                                       256, false, lds);
        for (const MtePlanTile& t : mte_plan_f32(jobs, 256, true, lds)) {
          CHECK(t.rows == rows);
          CHECK(t.waves == full[0].waves);
        }
      }
  // A launch that leaves CUs idle takes fewer rows, never fewer than 32 nor
  // more than the table's, and eight waves.
  for (int64_t N : {1, 100, 2000, 6000})
    for (int rows : {32, 64, 96, 128, 256}) {
      const auto p = mte_plan_f32({MtePlanJob{128, N, rows}}, 256, false, lds);
      CHECK(p[0].rows >= 32 && p[0].rows <= rows && p[0].rows % 32 == 0);
      if ((N + 31) / 32 <= 256) CHECK(p[0].rows == 32 || N / p[0].rows >= 256);
      if ((N + 31) / 32 <= 256) CHECK(p[0].waves == 8);
    }
  // One that fills them takes the table's rows, four waves up to 16 output
  // tiles of which two fit a CU's LDS.
  const auto f = mte_plan_f32({MtePlanJob{128, 100000, 128}, MtePlanJob{128, 100000, 256},
                               MtePlanJob{512, 100000, 32}, MtePlanJob{544, 100000, 32}},
                              256, false, lds);
  CHECK(f[0].rows == 128 && f[0].waves == 4);
  CHECK(f[1].rows == 256 && f[1].waves == 8);
  CHECK(f[2].rows == 32 && f[2].waves == 4);
  CHECK(f[3].rows == 32 && f[3].waves == 8);
  // Row scales: for noise that is there and small.
  const double prm[8] = {0.05, 0.05, 0.1, 0.5, 0.5, 0.05, 0.1, 0.2}, zero[8] = {};
  CHECK(!mte_low_noise(ROADMC_LAW_LOGNORMAL, 1.0, 0.0, prm));
  CHECK(mte_low_noise(ROADMC_LAW_LOGNORMAL, 1.0, 0.001, prm));
  CHECK(!mte_low_noise(ROADMC_LAW_LOGNORMAL, 1.0, 0.1, prm));
  CHECK(mte_low_noise(ROADMC_LAW_REF_CPU, 1.0, 0.0, prm));
  CHECK(!mte_low_noise(ROADMC_LAW_REF_CPU, 1.0, 0.1, zero));
  CHECK(mte_low_noise(ROADMC_LAW_REF_GPU, 1.0, 0.0, prm));
  CHECK(!mte_low_noise(ROADMC_LAW_REF_GPU, 1.0, 0.1, zero));
  printf("%s\n", failures ? "FAILED" : "ok");
  return failures ? 1 : 0;
}
