// kg_resident.hpp -- a whole small field in one work-group's LDS, many
// schedule steps to a launch.
//
// A field of a few thousand birds is far too little work for a launch per
// step: the tile kernels spend it on launch gaps and on one work-group's
// chain of global loads.  Here one work-group keeps every bird of a run in
// LDS for up to kResidentSteps schedule steps.  Each thread owns up to kB
// birds.  A step is: every thread walks its birds' windows in LDS into
// registers; then all birds are counted into bins (runs of 1 << shift rows
// of one column), the counts become starts, each bird's key (row, id) is
// ranked inside its bin, and the birds go back to LDS in bag-scan order.
// The last step's order is the read buffer's (tile by tile), so birds and
// bin offsets are written back as the other paths leave them.
//
// The neighbour sums take the near form (kg_near.hpp) while every bird is
// near, and full_step, the general form, in any step where one is not.
#pragma once

#include "kg_near.hpp"

namespace kg {

// Steps per launch.  A step of 4,096 birds takes 30 us where they are uniform
// at 0.025 per unit^2 and 1.5 ms in one blob of sigma 1 (a walk is linear in
// its window's birds, a step quadratic in a crowd's); the paths with a
// work-group per tile took 1.5 ms for that blob too.
constexpr uint32_t kResidentSteps = 256;
// What a work-group's registers and LDS hold.  Against the three-kernel path,
// fields of 0.025 birds per unit^2, us: one step 49 to 77 at 2,048 birds, 67
// to 75 at 4,096; 200 steps 2,999 to 3,942 at 2,048, 4,369 to 4,149 at 3,072,
// 5,971 to 4,494 at 4,096: single steps are shorter here at every size, runs
// of many up to about 2,900 birds.
constexpr uint32_t kResidentMaxAgents = 4096;
// z holds 12 bits of column here
constexpr int32_t kResidentMaxCols = 4095;
constexpr int32_t kResidentMaxRows = 1 << kNearRowBits;

// LDS of a run of up to `cap` birds and `bins` bins.
struct ResSmem {
  NearBirds b;    // cap; its records hold the keys while birds are in registers
  uint32_t* tab;  // bins + 1
};

KG_HD size_t res_smem_bytes(uint32_t cap, uint32_t bins) {
  return near_birds_bytes(cap) + (size_t)(bins + 1) * sizeof(uint32_t);
}

KG_HD ResSmem res_carve(uint8_t* p, uint32_t cap) {
  ResSmem s;
  s.b = near_birds_at(p, cap, &p);
  s.tab = (uint32_t*)p;
  return s;
}

// The field's own bins in LDS: columns of bins of 1 << shift rows, at most
// `bins` of them.
struct ResBins {
  int32_t rows, shift;  // bins per column
  uint32_t n;
};

KG_HD ResBins res_bins(const Geom& g, uint32_t bins) {
  ResBins b;
  b.shift = 0;
  while ((uint64_t)g.dw * (uint64_t)(((g.dh - 1) >> b.shift) + 1) > bins) ++b.shift;
  b.rows = ((g.dh - 1) >> b.shift) + 1;
  b.n = (uint32_t)(g.dw * b.rows);
  return b;
}

// Whether a run fits: `bins` receives the bin table it needs (at least the
// read buffer's bins, for the write-back, and one bin per column).
KG_HD bool res_fits(const RepDev& rp, uint32_t agents, size_t lds, uint32_t* bins) {
  const Geom& g = rp.g;
  if (!rp.lds_ok || agents == 0 || agents > kResidentMaxAgents || g.dw > kResidentMaxCols ||
      g.dh > kResidentMaxRows)
    return false;
  uint32_t b = agents > 1024u ? agents : 1024u;
  if (b < g.nbins) b = g.nbins;
  if (b < (uint32_t)g.dw) b = (uint32_t)g.dw;
  *bins = b;
  return res_smem_bytes(agents, b) <= lds;
}

// The runs of one launch: every work-group has the LDS of the most birds and
// of the largest bin table among them, which need not be one run's (4,096
// birds beside 200 in 16,384 bins: 163,868 bytes of a work-group's 163,840,
// where each alone takes less than 115,000).
struct ResGroup {
  uint32_t cap = 0, bins = 0;

  KG_HD void add(uint32_t agents, uint32_t res_bins) {
    cap = cap > agents ? cap : agents;
    bins = bins > res_bins ? bins : res_bins;
  }
  KG_HD bool fits(size_t lds) const { return res_smem_bytes(cap, bins) <= lds; }
};

// A bird between its walk and its place in LDS.
struct ResBird {
  float x, y, hx, hy;
  uint32_t id, z, bin, slot;
};

// Cell and bin of a bird; api: the read buffer's bins instead of the field's
// own.  A bird outside the grid is reported and kept in cell 0.
KG_HD void res_place(const RepDev& rp, const ResBins& rb, bool api, ResBird* b, uint32_t* err) {
  const Geom& g = rp.g;
  int32_t cx = cell_axis(g, b->x), cy = cell_axis(g, b->y);
  if (!cell_valid(g, cx, cy)) {
    atom_or(err, 1u);
    cx = cy = 0;
  }
  b->z = ((uint32_t)cx << kNearRowBits) | (uint32_t)cy;
  b->bin = api ? bin_of(g, cx, cy) : (uint32_t)(cx * rb.rows + (cy >> rb.shift));
}

KG_HD uint64_t res_key(const ResBird& b) {
  return ((uint64_t)(b.z & ((1u << kNearRowBits) - 1u)) << 32) | b.id;
}

// Bird::step of entry o in the general form (any toroidal field whose windows
// fit) from the same LDS layout.
template <class Find>
KG_HD void full_step(const RepDev& rp, uint64_t step, uint32_t o, const Find& find,
                     const NearBirds& B, NearRec* next) {
  const Geom& g = rp.g;
  const float T = rp.sq_thresh;
  const NearRec b = B.rec[o];
  const uint32_t id = B.id[o];
  const NearWindow w = near_window(rp, 0, (int32_t)(B.z[o] >> kNearRowBits),
                                   (int32_t)(B.z[o] & ((1u << kNearRowBits) - 1u)));
  FlockAcc acc;
  for (int32_t q = 0; q <= w.cols && w.rows >= 0; ++q) {
    uint32_t lo, hi;
    find.one(w.c + q, w.row, (uint32_t)w.rows, &lo, &hi);
    int32_t cur = -1;
    int chk = 0;
    for (uint32_t e = lo; e < hi; ++e) {
      const int32_t row = (int32_t)(B.z[e] & ((1u << kNearRowBits) - 1u));
      if (row != cur) {
        cur = row;
        chk = check_circle_sq(g, w.c + q, row, b.x, b.y, T);
      }
      if (chk == -1) continue;
      const NearRec c = B.rec[e];
      const float dx = toroidal_distance(b.x, c.x, g.w);
      const float dy = toroidal_distance(b.y, c.y, g.h);
      if (chk == 1 || dx * dx + dy * dy <= T) acc.add(B.id[e] == id, dx, dy, c.hx, c.hy);
    }
  }
  flock_finish(acc, rp.p, id, step, b.x, b.y, b.hx, b.hy, g.w, &next->x, &next->y, &next->hx,
               &next->hy);
}

}  // namespace kg
