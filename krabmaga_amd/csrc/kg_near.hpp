// kg_near.hpp -- Bird::step on "near" fields: toroidal fields whose windows
// never reach across the seam, which is every field more than a few cells
// wide.  There the reference's rules simplify exactly:
//
// - Two birds of one window lie within (dd + 1) cells of each other, at most
//   half the torus, so toroidal_distance is the plain difference.
// - check_circle's answer rarely matters.  A candidate within the radius is
//   returned unless all four corners of its cell are beyond it; on a field
//   whose cells are small against the radius (rep.sq_sure) some corner of
//   every window cell is always within it.  A candidate beyond the radius is
//   returned only if all four corners are within it, and then it lies at
//   most a few ulps beyond: only squared distances in (T, Tm] need the
//   corners looked at.
// - Quotients by a shared divisor take one reciprocal in f64 (recip_of).
//
// Every function gives the bits of the general form (kg_device.hpp).  A
// neighbourhood that holds a bird outside [0, w] x [0, h], a coordinate below
// 2^-60, a heading above 2^60 or a NaN is not near (near_bad); the caller
// takes the general form for it.
//
// The walk reads a list of birds in LDS sorted by z =
// column << kNearRowBits | row, then id: the reference's bag-scan order, in
// which the rows of one window column are one contiguous run.
#pragma once

#include "kg_phases.hpp"

namespace kg {

constexpr int kNearRowBits = 20;

struct alignas(16) NearRec {
  float x, y, hx, hy;
};

// Birds in scan order: bird e is rec[e] with key z[e] and id id[e]; one entry
// past the last has z = ~0u (its record is read, never used).
struct NearBirds {
  NearRec* rec;
  uint32_t* z;
  uint32_t* id;
};

KG_HD size_t near_birds_bytes(uint32_t n) {
  return (size_t)(n + 1) * (sizeof(NearRec) + 2 * sizeof(uint32_t));
}

// Birds [0, n] at p (16-byte aligned); *end: the first byte after them.
KG_HD NearBirds near_birds_at(uint8_t* p, uint32_t n, uint8_t** end) {
  NearBirds b;
  b.rec = (NearRec*)p;
  b.z = (uint32_t*)(b.rec + n + 1);
  b.id = b.z + n + 1;
  *end = (uint8_t*)(b.id + n + 1);
  return b;
}

KG_HD uint32_t f_bits(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __float_as_uint(v);
#else
  uint32_t u;
  __builtin_memcpy(&u, &v, 4);
  return u;
#endif
}

// Whether a bird takes its neighbourhood out of the near form.  (bits - 1)
// is huge for a zero of either sign: zeros are fine.
KG_HD bool near_bad(const Geom& g, float x, float y, float hx, float hy) {
  constexpr uint32_t kTiny = (127u - 60u) << 23;
  // false for NaN
  const bool in = x <= g.w && y <= g.h && fabsf(hx) <= 0x1p60f && fabsf(hy) <= 0x1p60f;
  return !in || f_bits(x) - 1u < kTiny - 1u || f_bits(y) - 1u < kTiny - 1u;
}

// 1 / b to 2^-52 relative, b a float with |b| in [2^-60, 2^81] (or 0, which
// gives NaN, as 0 / 0 does), for quot.  From the 2^-23 of v_rcp_f32, one
// third-order step: with e = 1 - b y, y (1 + e + e^2) is off by e^3.  f32
// division takes 45 cycles of a SIMD's issue per wave, quot 13 after 34 for
// the reciprocal (measured on MI355X, where f64 operations and conversions
// issue at the f32 rate).
KG_HD double recip_of(float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double d = (double)b;
  const double y = (double)__builtin_amdgcn_rcpf(b);
  const double e = __builtin_fma(-d, y, 1.0);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
#else
  return b == 0.0f ? (double)NAN : 1.0 / (double)b;
#endif
}

// Bird::step's neighbour sums (bird.rs:54-81); n counts the neighbours.
struct NearAcc {
  float x_avoid = 0.0f, y_avoid = 0.0f;
  float x_cohe = 0.0f, y_cohe = 0.0f;
  float x_cons = 0.0f, y_cons = 0.0f;
  int32_t n = 0;

  KG_HD void add(float dx, float dy, float square, float ehx, float ehy) {
    const double r = recip_of(square * square + 1.0f);
    n += 1;
    x_avoid += quot(dx, r);
    y_avoid += quot(dy, r);
    x_cohe += dx;
    y_cohe += dy;
    x_cons += ehx;
    y_cons += ehy;
  }
};

// check_circle (field_2d.rs:934-972) of cell (bx, by) for a bird at (lx, ly)
// with plain differences: all four corners within T (want = 1) or all four
// beyond it (want = -1); see window_checks for the two comparisons.
KG_HD bool near_corners(const Geom& g, int32_t bx, int32_t by, float lx, float ly, float T,
                        int want) {
  const float x0 = (float)bx * g.d, y0 = (float)by * g.d;
  // (no fminf: it would have the walk canonicalise g.w and g.h at every trip)
  const float xd = x0 + g.d, yd = y0 + g.d;
  const float x1 = xd < g.w ? xd : g.w, y1 = yd < g.h ? yd : g.h;
  const float ax = x0 - lx, bx2 = x1 - lx, ay = y0 - ly, by2 = y1 - ly;
  if (want == 1)
    return fmaxf(ax * ax, bx2 * bx2) + fmaxf(ay * ay, by2 * by2) <= T;
  return fminf(ax * ax, bx2 * bx2) + fminf(ay * ay, by2 * by2) > T;
}

// Candidate e of the bird `qid` at (qx, qy).
KG_HD void near_candidate(const RepDev& rp, int32_t col0, float qx, float qy, uint32_t qid,
                          const NearBirds& B, uint32_t e, const NearRec& c, uint32_t cid,
                          NearAcc* acc) {
  const float dx = qx - c.x, dy = qy - c.y;
  const float s = dx * dx + dy * dy;
  if (!((s <= rp.sq_near) & (cid != qid))) return;  // sq_sure <= sq_near
  if (!(s <= rp.sq_sure)) {  // rare: the corners decide
    const int32_t bx = col0 + (int32_t)(B.z[e] >> kNearRowBits);
    const int32_t by = (int32_t)(B.z[e] & ((1u << kNearRowBits) - 1u));
    const bool in = s <= rp.sq_thresh;
    if (near_corners(rp.g, bx, by, qx, qy, rp.sq_thresh, in ? -1 : 1) == in) return;
  }
  acc->add(dx, dy, s, c.hx, c.hy);
}

// Whether the bird at (qx, qy) of cell (cx, cy) finds itself: its own bag is
// in the window and not all of the bag's corners are beyond the radius.
KG_HD bool near_self(const RepDev& rp, float qx, float qy, int32_t cx, int32_t cy) {
  if (cx >= rp.g.max_x || cy >= rp.g.max_y) return false;
  return !(rp.sq_sure < 0.0f && near_corners(rp.g, cx, cy, qx, qy, rp.sq_thresh, -1));
}

// Whether every one of six sums is zero, infinite, NaN or at least 2^-60 in
// magnitude (doubling the bits drops the sign; minus one makes zero huge).
KG_HD uint32_t mag_key(float v) { return (f_bits(v) << 1) - 1u; }
KG_HD uint32_t umin2(uint32_t a, uint32_t b) { return a < b ? a : b; }
constexpr uint32_t kMagTiny = ((127u - 60u) << 24) - 1u;
constexpr uint32_t kMagHuge = ((127u + 60u) << 24) - 1u;

// bird.rs:83-153 with the shared reciprocals; flock_finish's arguments and
// results.  found: the neighbour vector is not empty.
KG_HD void near_finish(const NearAcc& a, bool found, const FlockParams& p, uint32_t id,
                       uint64_t step,
                       float px, float py, float hx, float hy, float width, float* nx, float* ny,
                       float* nhx, float* nhy) {
  const uint32_t m = umin2(umin2(umin2(mag_key(a.x_avoid), mag_key(a.y_avoid)),
                                 umin2(mag_key(a.x_cohe), mag_key(a.y_cohe))),
                           umin2(mag_key(a.x_cons), mag_key(a.y_cons)));
  const bool plain = m >= kMagTiny;
  float avoid_x = 0.0f, avoid_y = 0.0f, cohe_x = 0.0f, cohe_y = 0.0f;
  float rand_x = 0.0f, rand_y = 0.0f, cons_x = 0.0f, cons_y = 0.0f;
  if (found) {
    float x_avoid = a.x_avoid, y_avoid = a.y_avoid, x_cohe = a.x_cohe, y_cohe = a.y_cohe;
    cons_x = a.x_cons;
    cons_y = a.y_cons;
    if (a.n > 0) {
      const float c = (float)a.n;
      if (plain) {
        const double r = recip_of(c);
        x_avoid = quot(x_avoid, r);
        y_avoid = quot(y_avoid, r);
        x_cohe = quot(x_cohe, r);
        y_cohe = quot(y_cohe, r);
        cons_x = quot(quot(cons_x, r), r);
        cons_y = quot(quot(cons_y, r), r);
      } else {
        x_avoid /= c;
        y_avoid /= c;
        x_cohe /= c;
        y_cohe /= c;
        cons_x = cons_x / c / c;
        cons_y = cons_y / c / c;
      }
    }
    avoid_x = 400.0f * x_avoid;
    avoid_y = 400.0f * y_avoid;
    if (plain) {
      // 0.1 is off by 2^-56 relative: the same argument as recip_of's
      cohe_x = quot(-x_cohe, 0.1);
      cohe_y = quot(-y_cohe, 0.1);
    } else {
      cohe_x = -x_cohe / 10.0f;
      cohe_y = -y_cohe / 10.0f;
    }
    float r1, r2;
    step_uniforms(p.seed, id, step, &r1, &r2);
    const float x_rand = r1 * 2.0f - 1.0f;
    const float y_rand = r2 * 2.0f - 1.0f;
    // the draws are multiples of 2^-23: sq is zero or at least that
    const float sq = sqrtf(x_rand * x_rand + y_rand * y_rand);
    const double rs = recip_of(sq);
    rand_x = quot(0.05f * x_rand, rs);
    rand_y = quot(0.05f * y_rand, rs);
  }
  float dx = p.cohesion * cohe_x + p.avoidance * avoid_x + p.consistency * cons_x +
             p.randomness * rand_x + p.momentum * hx;
  float dy = p.cohesion * cohe_y + p.avoidance * avoid_y + p.consistency * cons_y +
             p.randomness * rand_y + p.momentum * hy;
  const float dis = sqrtf(dx * dx + dy * dy);
  if (dis > 0.0f) {
    if (umin2(mag_key(dx), mag_key(dy)) >= kMagTiny && mag_key(dis) >= kMagTiny &&
        mag_key(dis) < kMagHuge) {
      const double r = recip_of(dis);
      dx = quot(dx, r) * p.jump;
      dy = quot(dy, r) * p.jump;
    } else {
      dx = dx / dis * p.jump;
      dy = dy / dis * p.jump;
    }
  }
  *nhx = dx;
  *nhy = dy;
  // |dx|, |dy| <= 1.5 |jump| <= 0.45 width and py <= 1.5 width, or both NaN:
  // toroidal_transform without its fmod case
  const float vx = px + dx, vy = py + dy;  // bird.rs:147 wraps y by width
  *nx = vx >= width ? vx - width : (vx < 0.0f ? vx + width : vx);
  *ny = vy >= width ? vy - width : (vy < 0.0f ? vy + width : vy);
}

// First entry of z[lo, hi) at or after key.
KG_HD uint32_t near_lower(const uint32_t* z, uint32_t lo, uint32_t hi, uint32_t key) {
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (z[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Where a window column's run lies: entries [lo, hi) have z in [key, key +
// rows], key = c << kNearRowBits | row; of one column, or of up to three
// neighbouring ones (those past `cols` are empty).
//
// TileFind: the birds are the staged columns of a tile, column c from
// col_base[c] - base; both ends of a column's run bisected.
struct TileFind {
  const uint32_t* z;
  const uint32_t* col_base;
  uint32_t base;

  KG_HD void one(int32_t c, int32_t row, uint32_t rows, uint32_t* lo, uint32_t* hi) const {
    const uint32_t key = ((uint32_t)c << kNearRowBits) + (uint32_t)row;
    const uint32_t end = col_base[c + 1] - base;
    *lo = near_lower(z, col_base[c] - base, end, key);
    *hi = near_lower(z, *lo, end, key + rows + 1u);
  }
};

// StripFind: the same birds with the strips' starts (near_strips): a run's
// ends are at most a strip from a table entry, and where strips are single
// rows they are entries.  Bisecting and stepping were a fifth of the
// instructions of a dense tile (a round of 512 birds 6.6 us, 2.9 of them
// here).
struct StripFind : TileFind {
  const uint16_t* strip;
  int32_t n, per, sh, y0;

  KG_HD void three(int32_t c, int32_t cols, int32_t row, uint32_t rows, uint32_t* lo,
                   uint32_t* hi) const {
    const int32_t r0 = row - y0, r1 = r0 + (int32_t)rows;
    const int32_t j0 = imin(imax(r0 >> sh, -1), n) + 1, j1 = imin(imax(r1 >> sh, -1), n) + 1;
    const uint16_t* const s0 = strip + c * per;
    if (sh == 0) {  // single rows (and bands of one: three() is for disc_dist = 1)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        lo[q] = q <= cols ? s0[q * per + j0] - base : 0u;
        hi[q] = q <= cols ? s0[q * per + j1 + 1] - base : 0u;
      }
      return;
    }
    const uint32_t key = ((uint32_t)c << kNearRowBits) + (uint32_t)row;
    uint32_t first[3], last[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lo[q] = q <= cols ? s0[q * per + j0] - base : 0u;
      hi[q] = q <= cols ? s0[q * per + j1] - base : 0u;
      first[q] = q <= cols ? key + ((uint32_t)q << kNearRowBits) : 0u;
      last[q] = q <= cols ? first[q] + rows : 0u;
    }
    // both sides of each condition: no branch; the sentinel ends every run
    for (bool more = true; more;) {
      more = false;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bool before = z[lo[q]] < first[q];
        lo[q] += before ? 1u : 0u;
        more |= before;
      }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) hi[q] = hi[q] < lo[q] ? lo[q] : hi[q];
    for (bool more = true; more;) {
      more = false;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bool in = (z[hi[q]] <= last[q]) & (q <= cols);
        hi[q] += in ? 1u : 0u;
        more |= in;
      }
    }
  }
};

// CellFind: the birds are a whole field in bins of 1 << shift rows, column by
// column, `per` bins to a column, bin b from start[b].
struct CellFind {
  const uint32_t* z;
  const uint32_t* start;
  int32_t per, shift;

  KG_HD void one(int32_t c, int32_t row, uint32_t rows, uint32_t* lo, uint32_t* hi) const {
    const int32_t b0 = c * per + (row >> shift);
    const int32_t b1 = c * per + ((row + (int32_t)rows) >> shift);
    *lo = start[b0];
    if (shift == 0) {
      *hi = start[b1 + 1];
      return;
    }
    const uint32_t key = ((uint32_t)c << kNearRowBits) + (uint32_t)row;
    while (z[*lo] < key) ++*lo;  // the last entry's z is ~0u
    *hi = start[b1] > *lo ? start[b1] : *lo;
    while (z[*hi] <= key + rows) ++*hi;
  }
  KG_HD void three(int32_t c, int32_t cols, int32_t row, uint32_t rows, uint32_t* lo,
                   uint32_t* hi) const {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lo[q] = hi[q] = 0u;
      if (q <= cols) one(c + q, row, rows, &lo[q], &hi[q]);
    }
  }
};

// The clamped window of a bird in cell (c + col0, cy) (field_2d.rs:401-416),
// columns relative to col0; empty if cols < 0 or rows < 0.
struct NearWindow {
  int32_t c, cols, row, rows;
};

KG_HD NearWindow near_window(const RepDev& rp, int32_t col0, int32_t c, int32_t cy) {
  const int32_t dd = rp.disc_dist;
  NearWindow w;
  w.c = imax(-col0, c - dd);
  w.cols = imin(c + dd, rp.g.max_x - 1 - col0) - w.c;
  w.row = imax(0, cy - dd);
  w.rows = imin(cy + dd, rp.g.max_y - 1) - w.row;
  return w;
}

// Entry of candidate k of three runs of n0, n1 - n0 and the rest, from o0, o1
// + n0 and o2 + n1 (by value: two selects, no memory).
KG_HD uint32_t near_at(uint32_t k, uint32_t n0, uint32_t n1, uint32_t o0, uint32_t o1,
                       uint32_t o2) {
  uint32_t o = k < n1 ? o1 : o2;
  o = k < n0 ? o0 : o;
  return k + o;
}

// The neighbour sums of the bird `qid` at (qx, qy) over window w.  kFlat: one
// loop over the runs of three columns, else a loop per column (cheaper per
// candidate where every run is long).  Two candidates to a trip, the next one
// loaded while one is worked on.
template <bool kFlat, class Find>
KG_HD void near_walk(const RepDev& rp, int32_t col0, const NearWindow& w, float qx, float qy,
                     uint32_t qid, const Find& find, const NearBirds& B, NearAcc* acc) {
  if (w.cols < 0 || w.rows < 0) return;
  const uint32_t rows = (uint32_t)w.rows;
  if constexpr (kFlat) {
    if (rp.disc_dist == 1) {
      // a wave's trips are those of its busiest lane, not of each column's
      uint32_t lo[3], hi[3];
      find.three(w.c, w.cols, w.row, rows, lo, hi);
      const uint32_t n0 = hi[0] - lo[0], n1 = n0 + hi[1] - lo[1], n = n1 + hi[2] - lo[2];
      const uint32_t o1 = lo[1] - n0, o2 = lo[2] - n1;
      const uint32_t o0 = lo[0];
      if (n == 0u) return;
      uint32_t e = near_at(0u, n0, n1, o0, o1, o2), k = 0;
      NearRec c = B.rec[e];
      uint32_t id = B.id[e];
      for (; k + 1u < n; k += 2) {
        const uint32_t e1 = near_at(k + 1u, n0, n1, o0, o1, o2);
        const NearRec c1 = B.rec[e1];
        const uint32_t id1 = B.id[e1];
        near_candidate(rp, col0, qx, qy, qid, B, e, c, id, acc);
        // past the last candidate this is at most the sentinel
        e = near_at(k + 2u, n0, n1, o0, o1, o2);
        c = B.rec[e];
        id = B.id[e];
        near_candidate(rp, col0, qx, qy, qid, B, e1, c1, id1, acc);
      }
      if (k < n) near_candidate(rp, col0, qx, qy, qid, B, e, c, id, acc);
      return;
    }
  }
  for (int32_t q = 0; q <= w.cols; ++q) {
    uint32_t lo, hi;
    find.one(w.c + q, w.row, rows, &lo, &hi);
    if (lo >= hi) continue;
    NearRec c = B.rec[lo];
    uint32_t id = B.id[lo], e = lo;
    for (; e + 1u < hi; e += 2) {
      const NearRec c1 = B.rec[e + 1u];
      const uint32_t id1 = B.id[e + 1u];
      near_candidate(rp, col0, qx, qy, qid, B, e, c, id, acc);
      c = B.rec[e + 2u];  // at most the sentinel
      id = B.id[e + 2u];
      near_candidate(rp, col0, qx, qy, qid, B, e + 1u, c1, id1, acc);
    }
    if (e < hi) near_candidate(rp, col0, qx, qy, qid, B, e, c, id, acc);
  }
}

// Whether the window holds any bird the query returns (near_walk skips those
// with the own id): for a bird that does not find itself.
template <class Find>
KG_HD bool near_any(const RepDev& rp, int32_t col0, const NearWindow& w, float qx, float qy,
                    const Find& find, const NearBirds& B) {
  for (int32_t q = 0; q <= w.cols && w.rows >= 0; ++q) {
    uint32_t lo, hi;
    find.one(w.c + q, w.row, (uint32_t)w.rows, &lo, &hi);
    for (uint32_t e = lo; e < hi; ++e) {
      const float dx = qx - B.rec[e].x, dy = qy - B.rec[e].y;
      const float s = dx * dx + dy * dy;
      const bool in = s <= rp.sq_thresh;
      const int32_t by = (int32_t)(B.z[e] & ((1u << kNearRowBits) - 1u));
      const bool flip = s > rp.sq_sure && s <= rp.sq_near &&
                        near_corners(rp.g, col0 + w.c + q, by, qx, qy, rp.sq_thresh, in ? -1 : 1);
      if (in != flip) return true;
    }
  }
  return false;
}

// Bird::step of entry o.
template <bool kFlat, class Find>
KG_HD void near_step(const RepDev& rp, int32_t col0, uint64_t step, uint32_t o, const Find& find,
                     const NearBirds& B, NearRec* next) {
  const NearRec b = B.rec[o];
  const uint32_t z = B.z[o], id = B.id[o];
  const int32_t c = (int32_t)(z >> kNearRowBits);
  const int32_t cy = (int32_t)(z & ((1u << kNearRowBits) - 1u));
  const NearWindow w = near_window(rp, col0, c, cy);
  NearAcc acc;
  near_walk<kFlat>(rp, col0, w, b.x, b.y, id, find, B, &acc);
  bool found = acc.n != 0 || near_self(rp, b.x, b.y, col0 + c, cy);
  if (!found) found = near_any(rp, col0, w, b.x, b.y, find, B);
  near_finish(acc, found, rp.p, id, step, b.x, b.y, b.hx, b.hy, rp.g.w, &next->x, &next->y,
              &next->hx, &next->hy);
}

// ---- staging a tile ---------------------------------------------------------
//
// A tile's own birds are one run of the read buffer, so they are enumerated
// by their read-buffer index; the halo's (the bands above and below the own
// columns, whole columns beside them) follow.  Both go to their place in the
// z order.

// Where the strips of a tile's staged columns start: a column's entries are
// the band below the tile, its own rows in strips of 1 << sh rows (whole bins,
// whose starts the read buffer's offsets give), the band above, and its end.
// As many strips to a column as kNearStrips entries allow (one strip always
// fits: kMaxStageCols columns of 4).
constexpr int kNearStrips = 4 * kMaxStageCols;

struct NearStrips {
  int32_t n, per, sh;  // strips of a column, its entries (n + 3), rows of a strip (log2)
};

KG_HD NearStrips near_strips(const RepDev& rp) {
  const Geom& g = rp.g;
  const int32_t cols = imin(kMaxStageCols, g.tx + 2 * rp.disc_dist);
  int32_t up = 0;
  while ((g.tr >> up) > 1 && cols * ((g.tr >> up) + 3) > kNearStrips) ++up;
  return NearStrips{g.tr >> up, (g.tr >> up) + 3, g.hb_log2 + up};
}

// LDS of a staged tile: `cap` birds and the per-column tables of `cols`
// columns.
struct NearSmem {
  NearBirds b;          // cap
  uint32_t* seg_start;  // 3 per column (flock_segments)
  uint32_t* seg_len;    // 3 per column
  uint32_t* col_base;   // cols + 1
  uint16_t* own;        // cap: slots of the own birds, in read-buffer order
  uint16_t* strip;      // kNearStrips (near_strips)
};

KG_HD size_t near_smem_bytes(int cap, int cols) {
  return near_birds_bytes((uint32_t)cap) + (size_t)(7 * cols + 1) * sizeof(uint32_t) +
         (size_t)(((cap + 1) & ~1) + kNearStrips) * sizeof(uint16_t);
}

KG_HD NearSmem near_carve(uint8_t* p, int cap, int cols) {
  NearSmem s;
  s.b = near_birds_at(p, (uint32_t)cap, &p);
  s.seg_start = (uint32_t*)p;
  s.seg_len = s.seg_start + 3 * cols;
  s.col_base = s.seg_len + 3 * cols;
  s.own = (uint16_t*)(s.col_base + cols + 1);
  s.strip = s.own + ((cap + 1) & ~1);
  return s;
}

// The staged items of own columns [oa, ob): staged columns [sa, sb), n items
// of which nown are the own birds [own_lo, own_lo + nown) of the read buffer.
struct NearChunk {
  int32_t oa, ob, sa, sb;
  uint32_t base, n, own_lo, nown;
};

KG_HD NearChunk near_chunk(const RepDev& rp, const FlockTile& ft, const NearSmem& S, int32_t oa,
                           int32_t ob) {
  NearChunk k;
  k.oa = oa;
  k.ob = ob;
  flock_chunk_cols(rp, ft, oa, ob, &k.sa, &k.sb);
  k.base = S.col_base[k.sa];
  k.n = S.col_base[k.sb] - k.base;
  k.own_lo = S.seg_start[3 * oa + 1];
  k.nown = S.seg_start[3 * (ob - 1) + 1] + S.seg_len[3 * (ob - 1) + 1] - k.own_lo;
  return k;
}

// Halo items in staged columns [sa, c).
KG_HD uint32_t near_halo_before(const NearChunk& k, const NearSmem& S, int32_t c) {
  const uint32_t all = S.col_base[c] - k.base;
  if (c <= k.oa) return all;
  return all - (c >= k.ob ? k.nown : S.seg_start[3 * c + 1] - k.own_lo);
}

// Read-buffer index of halo item m, and its slot.
KG_HD uint32_t near_halo(const NearChunk& k, const NearSmem& S, uint32_t m, uint32_t* slot) {
  int32_t lo = k.sa, hi = k.sb;  // column c with before(c) <= m < before(c + 1)
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (near_halo_before(k, S, mid) <= m) lo = mid;
    else hi = mid;
  }
  uint32_t off = m - near_halo_before(k, S, lo);
  const uint32_t l0 = S.seg_len[3 * lo], l1 = S.seg_len[3 * lo + 1];
  const uint32_t first = S.col_base[lo] - k.base;
  if (off < l0) {
    *slot = first + off;
    return S.seg_start[3 * lo] + off;
  }
  off -= l0;
  if (lo < k.oa || lo >= k.ob) {
    if (off < l1) {
      *slot = first + l0 + off;
      return S.seg_start[3 * lo + 1] + off;
    }
    off -= l1;
  }
  *slot = first + l0 + l1 + off;
  return S.seg_start[3 * lo + 2] + off;
}

// Stages item i (< k.n: own birds first); false if it is not near.
KG_HD bool near_stage(const RepDev& rp, const FlockTile& ft, const NearChunk& k, uint32_t i,
                      Buf R, const NearSmem& S) {
  const Geom& g = rp.g;
  uint32_t slot = 0, gi;
  const bool mine = i < k.nown;
  if (mine) gi = k.own_lo + i;
  else gi = near_halo(k, S, i - k.nown, &slot);
  const float x = R.x[gi], y = R.y[gi];
  const float hx = R.hx[gi], hy = R.hy[gi];
  const uint32_t id = R.id[gi];
  const int32_t c = cell_axis(g, x) - ft.sc_lo;
  const int32_t cy = cell_axis(g, y);
  if (mine) {
    slot = S.col_base[c] - k.base + S.seg_len[3 * c] + (gi - S.seg_start[3 * c + 1]);
    S.own[i] = (uint16_t)slot;
  }
  S.b.rec[slot] = NearRec{x, y, hx, hy};
  S.b.z[slot] = ((uint32_t)c << kNearRowBits) | (uint32_t)cy;
  S.b.id[slot] = id;
  return !near_bad(g, x, y, hx, hy);
}

// Whether staged item i of a chunk is near (without staging it).
KG_HD bool near_item_ok(const RepDev& rp, const NearChunk& k, uint32_t i, Buf R,
                        const NearSmem& S) {
  uint32_t slot;
  const uint32_t gi = i < k.nown ? k.own_lo + i : near_halo(k, S, i - k.nown, &slot);
  return !near_bad(rp.g, R.x[gi], R.y[gi], R.hx[gi], R.hy[gi]);
}

// Entry i (< ft.ncols * near_strips().per) of the strips' table, counted from
// the tile's first staged bird (col_base).
KG_HD void near_strip_fill(const RepDev& rp, const FlockTile& ft, const NearStrips& st, uint32_t i,
                           const uint32_t* offset, const NearSmem& S) {
  const Geom& g = rp.g;
  const int32_t c = (int32_t)(i / (uint32_t)st.per), j = (int32_t)(i % (uint32_t)st.per) - 1;
  uint32_t v = S.col_base[c];
  if (j > st.n) {
    v = S.col_base[c + 1];
  } else if (j >= 0) {
    v += S.seg_len[3 * c];
    if (j == st.n) {
      v += S.seg_len[3 * c + 1];
    } else if (S.seg_len[3 * c + 1] != 0u) {
      const int32_t col = ft.sc_lo + c;
      const uint32_t tt = (uint32_t)(ft.tcy * g.ntx + (col >> g.tx_log2));
      const uint32_t b = rp.bin_base + col_bin0(g, tt, col & (g.tx - 1)) +
                         ((uint32_t)j << (st.sh - g.hb_log2));
      v += offset[b] - S.seg_start[3 * c + 1];
    }
  }
  S.strip[i] = (uint16_t)v;
}

// Bird::step of own bird o of a staged chunk.
KG_HD void near_agent(const RepDev& rp, const FlockTile& ft, const NearChunk& k,
                      const NearStrips& st, uint32_t o, const NearSmem& S, Buf W,
                      uint32_t* count_next, uint32_t* err, const FlockSinks& lv) {
  NearRec r;
  const StripFind find{{S.b.z, S.col_base, k.base}, S.strip, st.n, st.per, st.sh, ft.y0};
  near_step<true>(rp, ft.sc_lo, ft.step, S.own[o], find, S.b, &r);
  flock_emit(rp.g, rp.bin_base, W, k.own_lo + o, r.x, r.y, r.hx, r.hy, count_next, err, ft.tile,
             lv);
}

// ---- staging a run of birds ---------------------------------------------------
//
// A tile too full for LDS is stepped by runs of its birds, each with only its
// own neighbourhood staged: the columns the run's windows reach, whole tile
// height if the run spans columns, else the rows around its own.  A run of a
// dense column is a dozen rows, so three short column pieces hold its
// neighbours.

// LDS of a piece (a tile's without the own list).
KG_HD size_t near_piece_bytes(int cap, int cols) {
  return near_birds_bytes((uint32_t)cap) + (size_t)(7 * cols + 1) * sizeof(uint32_t);
}

// The staged rectangle of birds that lie in columns [ca, cb], rows [r0, r1] of
// tile ft: ft with its staged columns and rows replaced.
KG_HD FlockTile near_piece(const RepDev& rp, FlockTile ft, int32_t ca, int32_t cb, int32_t r0,
                           int32_t r1) {
  const Geom& g = rp.g;
  const int32_t dd = rp.disc_dist;
  ft.sc_lo = imax(0, ca - dd);
  ft.ncols = imax(cb, imin(g.max_x - 1, cb + dd)) - ft.sc_lo + 1;
  ft.ry_lo = imax(0, r0 - dd);
  ft.ry_hi = imax(r1, imin(g.max_y - 1, r1 + dd));
  return ft;
}

// Stages item i (< col_base[ncols]) of a piece at slot i; false if it is not
// near.
KG_HD bool near_stage_piece(const RepDev& rp, const FlockTile& pt, uint32_t i, Buf R,
                            const NearSmem& S) {
  int32_t lo = 0, hi = pt.ncols;  // column c with col_base[c] <= i < col_base[c + 1]
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (S.col_base[mid] <= i) lo = mid;
    else hi = mid;
  }
  uint32_t off = i - S.col_base[lo];
  const uint32_t l0 = S.seg_len[3 * lo], l1 = S.seg_len[3 * lo + 1];
  uint32_t gi = S.seg_start[3 * lo] + off;
  if (off >= l0 + l1) gi = S.seg_start[3 * lo + 2] + (off - l0 - l1);
  else if (off >= l0) gi = S.seg_start[3 * lo + 1] + (off - l0);
  const NearRec r{R.x[gi], R.y[gi], R.hx[gi], R.hy[gi]};
  S.b.rec[i] = r;
  S.b.z[i] = ((uint32_t)lo << kNearRowBits) | (uint32_t)cell_axis(rp.g, r.y);
  S.b.id[i] = R.id[gi];
  return !near_bad(rp.g, r.x, r.y, r.hx, r.hy);
}

// Bird::step of read-buffer bird gi of a staged piece.
KG_HD void near_agent_piece(const RepDev& rp, const FlockTile& pt, uint32_t gi, Buf R,
                            const NearSmem& S, Buf W, uint32_t* count_next, uint32_t* err,
                            const FlockSinks& lv) {
  const int32_t c = cell_axis(rp.g, R.x[gi]) - pt.sc_lo;
  const uint32_t slot = S.col_base[c] + S.seg_len[3 * c] + (gi - S.seg_start[3 * c + 1]);
  NearRec r;
  near_step<false>(rp, pt.sc_lo, pt.step, slot, TileFind{S.b.z, S.col_base, 0u}, S.b, &r);
  flock_emit(rp.g, rp.bin_base, W, gi, r.x, r.y, r.hx, r.hy, count_next, err, pt.tile, lv);
}

}  // namespace kg
