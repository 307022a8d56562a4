// group_check.cpp -- which runs may share a launch of the resident step
// (kg_resident.hpp, ResGroup): a launch gives every work-group the LDS of the
// most birds and of the largest bin table among its runs, so runs that fit
// alone may not fit together.  Exit status 0: every scenario agrees.
#include <cstdio>
#include <random>
#include <vector>

#include "kg_geom.hpp"
#include "kg_resident.hpp"

using namespace kg;

// 160 KB of a work-group less the static LDS the host sets aside.
constexpr size_t kLds = 160 * 1024 - 6144;

struct Run {
  uint32_t n;
  float w, h;
  uint32_t tx, ty, hb;
};

// The run's bin table and device bins; 0 if it does not fit alone.
static uint32_t bins_of(const Run& r, uint32_t* nbins) {
  RepDev rp{};
  std::string why;
  if (!make_geom_rt(r.w, r.h, 10.0f / 1.5f, 1, r.n, r.tx, r.ty, r.hb, &rp.g, &why)) return 0;
  kg_flock_params p{1, 1, 1, 1, 1, 0.7f, 10.0f, 0, 0};
  set_rep_params(&rp, p);
  *nbins = rp.g.nbins;
  uint32_t b = 0;
  return res_fits(rp, r.n, kLds, &b) ? b : 0u;
}

// A group fits exactly when its launch fits LDS and has room for every run.
static int check(const char* name, const std::vector<Run>& runs, int want) {
  ResGroup grp;
  std::vector<uint32_t> nbins(runs.size());
  for (size_t i = 0; i < runs.size(); ++i) {
    const uint32_t b = bins_of(runs[i], &nbins[i]);
    if (!b) {
      std::printf("%s: run %zu does not fit alone\n", name, i);
      return 1;
    }
    grp.add(runs[i].n, b);
  }
  const bool fits = grp.fits(kLds);
  bool room = true;
  for (size_t i = 0; i < runs.size(); ++i) room = room && runs[i].n <= grp.cap && nbins[i] <= grp.bins;
  const bool launch = res_smem_bytes(grp.cap, grp.bins) <= kLds;
  if (!room || fits != launch || (want >= 0 && fits != (want != 0))) {
    std::printf("%s: fits %d, launch of %zu bytes\n", name, fits,
                res_smem_bytes(grp.cap, grp.bins));
    return 1;
  }
  std::printf("%s: %u birds, %u bins, %zu bytes: %s\n", name, grp.cap, grp.bins,
              res_smem_bytes(grp.cap, grp.bins), fits ? "one launch" : "not one launch");
  return 0;
}

int main() {
  int failed = 0;
  const Run full{4096, 404.8f, 404.8f, 0, 0, 0};
  failed += check("one full run", {full}, 1);
  failed += check("two full runs", {full, full}, 1);
  failed += check("full and small", {full, {1000, 200, 200, 0, 0, 0}}, 1);
  failed += check("full and sparse", {full, {200, 27000, 27000, 0, 0, 0}}, 0);
  failed += check("full and wide", {full, {500, 26667, 40000, 0, 0, 0}}, 0);
  failed += check("small bins", {{4096, 404.8f, 404.8f, 8, 32, 1}, {500, 1000, 1000, 8, 32, 1}}, 0);
  failed += check("small and sparse", {{1000, 200, 200, 0, 0, 0}, {200, 27000, 27000, 0, 0, 0}}, 1);
  std::mt19937 rng(7);
  int groups = 0;
  for (int k = 0; k < 400; ++k) {
    std::vector<Run> runs;
    for (int i = 0; i < 4; ++i) {
      const uint32_t n = 1 + rng() % 4096;
      const float side = 50.0f + (float)(rng() % 30000);
      Run r{n, side, side, 0, 0, 0};
      uint32_t nb = 0;
      if (bins_of(r, &nb)) runs.push_back(r);
    }
    if (runs.size() < 2) continue;
    ++groups;
    failed += check("random", runs, -1);
  }
  if (groups < 100) ++failed;
  std::printf("%d scenario(s) failed\n", failed);
  return failed ? 1 : 0;
}
