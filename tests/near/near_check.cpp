// near_check.cpp -- the near form of Bird::step (kg_near.hpp) against the
// general form (flock_agent_global) on the CPU, bit for bit, tile by tile as
// k_flock_near stages them.  Exit status 0: every scenario agrees.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "kg_geom.hpp"
#include "kg_near.hpp"

using namespace kg;

struct Case {
  const char* name;
  uint32_t n;
  float w, h, d, radius, jump;
  uint32_t tx, ty, hb;
  int cap;       // birds staged at once
  int layout;    // 0 uniform, 1 cell corners, 2 one crowded spot, 3 on the far edges
  int headings;  // 0 unit, 1 tiny and zero, 2 infinite and NaN now and then
  float wt;      // cohesion and avoidance weight
  bool near;     // whether the near form must apply
};

struct Cols {
  std::vector<float> x, y, hx, hy;
  std::vector<uint32_t> id;
  explicit Cols(size_t n) : x(n), y(n), hx(n), hy(n), id(n) {}
  Buf view() { return Buf{x.data(), y.data(), hx.data(), hy.data(), id.data()}; }
};

static bool same(float a, float b) {
  if (a != a && b != b) return true;
  return std::memcmp(&a, &b, 4) == 0;
}

static int run(const Case& c, uint64_t seed) {
  Geom g{};
  std::string why;
  if (!make_geom_rt(c.w, c.h, c.d, 1, c.n, c.tx, c.ty, c.hb, &g, &why)) {
    std::printf("%s: %s\n", c.name, why.c_str());
    return 1;
  }
  RepDev rp{};
  rp.g = g;
  kg_flock_params p{c.wt, c.wt, 1.3f, 0.7f, 0.9f, c.jump, c.radius, 0u, seed};
  set_rep_params(&rp, p);
  rp.step_base = 3;
  if ((rp.near != 0) != c.near) {
    std::printf("%s: near is %d\n", c.name, rp.near);
    return 1;
  }
  if (!rp.near) return 0;
  std::mt19937_64 rng(seed * 7919 + c.n);
  auto u = [&] { return (float)(rng() >> 40) * 0x1p-24f; };
  Cols A(c.n);
  for (uint32_t i = 0; i < c.n; ++i) {
    float x = c.w * u(), y = c.h * u();
    if (c.layout == 1) {  // on and one ulp around the corners of cells
      x = (float)(rng() % (uint64_t)g.max_x) * c.d;
      y = (float)(rng() % (uint64_t)g.max_y) * c.d;
      if (rng() % 3 == 0) x = std::nextafter(x, c.w);
      if (rng() % 3 == 0) y = std::nextafter(y, 0.0f);
    } else if (c.layout == 2 && i % 2) {
      x = c.w * 0.37f + 3.0f * u();
      y = c.h * 0.61f + 3.0f * u();
    } else if (c.layout == 3 && i % 4 == 0) {
      if (rng() % 2) x = c.w;
      else y = c.h;
    }
    int32_t cx, cy;
    discretize(g, x, y, &cx, &cy);
    if (!cell_valid(g, cx, cy)) x = y = 0.0f;
    A.x[i] = x;
    A.y[i] = y;
    const float a = 6.2831853f * u();
    A.hx[i] = std::cos(a);
    A.hy[i] = std::sin(a);
    if (c.headings == 1) {
      A.hx[i] = rng() % 2 ? 1e-38f * u() : 0.0f;
      A.hy[i] = rng() % 2 ? -1e-25f * u() : 0.0f;
    } else if (c.headings == 2) {
      if (rng() % 3000 == 0) A.hx[i] = INFINITY;
      if (rng() % 3000 == 0) A.hy[i] = NAN;
      if (rng() % 50 == 0) A.hx[i] *= 1e17f;
    }
    A.id[i] = rng() % 40 ? i : i / 2;  // a few equal ids
  }
  // the binned read buffer
  std::vector<uint32_t> ord(c.n), bin(c.n);
  std::vector<int32_t> row(c.n);
  for (uint32_t i = 0; i < c.n; ++i) {
    int32_t cx;
    discretize(g, A.x[i], A.y[i], &cx, &row[i]);
    bin[i] = bin_of(g, cx, row[i]);
    ord[i] = i;
  }
  std::sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) {
    if (bin[a] != bin[b]) return bin[a] < bin[b];
    if (row[a] != row[b]) return row[a] < row[b];
    if (A.id[a] != A.id[b]) return A.id[a] < A.id[b];
    return a < b;
  });
  Cols R(c.n), W(c.n), V(c.n);
  std::vector<uint32_t> offset(g.nbins + 1, 0u);
  for (uint32_t k = 0; k < c.n; ++k) {
    const uint32_t i = ord[k];
    R.x[k] = A.x[i];
    R.y[k] = A.y[i];
    R.hx[k] = A.hx[i];
    R.hy[k] = A.hy[i];
    R.id[k] = A.id[i];
    ++offset[bin[i] + 1];
  }
  for (uint32_t b = 0; b < g.nbins; ++b) offset[b + 1] += offset[b];
  std::vector<uint32_t> cnt(g.nbins, 0u), want(g.nbins, 0u);
  uint32_t err = 0, err2 = 0;
  const uint32_t prefix[2] = {0u, g.ntiles};
  const int cols = std::min(kMaxStageCols, g.tx + 2 * rp.disc_dist);
  std::vector<uint64_t> smem((near_smem_bytes(c.cap, cols) + 7) / 8 + 2);
  uint32_t stepped = 0, chunks = 0, bad_tiles = 0;
  for (uint32_t item = 0; item < g.ntiles; ++item) {
    const FlockTile ft = flock_tile(&rp, 1, prefix, item, 0);
    uint8_t* base = (uint8_t*)(((uintptr_t)smem.data() + 15) & ~(uintptr_t)15);
    const NearSmem S = near_carve(base, c.cap, cols);
    uint32_t L = 0;
    for (int t = 0; t < ft.ncols; ++t) {
      S.col_base[t] = L;
      L += flock_segments(rp, ft, t, offset.data(), S.seg_start, S.seg_len);
    }
    S.col_base[ft.ncols] = L;
    const NearStrips st = near_strips(rp);
    if (ft.ncols * st.per > kNearStrips) return 1;
    for (uint32_t i = 0; i < (uint32_t)(ft.ncols * st.per); ++i)
      near_strip_fill(rp, ft, st, i, offset.data(), S);
    const int32_t lo = ft.c0 - ft.sc_lo, hi = ft.c1 - ft.sc_lo;
    const uint32_t cap = (uint32_t)c.cap;
    bool fits = true;
    for (int32_t q = lo; q < hi; ++q)
      if (flock_chunk_size(rp, ft, S.col_base, q, q + 1) > cap) fits = false;
    if (!fits) continue;
    const NearChunk all = near_chunk(rp, ft, S, lo, hi);
    bool ok = true;
    for (uint32_t i = 0; i < all.n; ++i)
      if (!near_item_ok(rp, all, i, R.view(), S)) ok = false;
    if (!ok) {
      ++bad_tiles;
      continue;
    }
    const FlockSinks lv{Outbox{}, 0u, nullptr, nullptr, nullptr};
    for (int32_t oa = lo; oa < hi;) {
      const int32_t ob = L > cap ? flock_chunk_end(rp, ft, S.col_base, oa, hi, cap) : hi;
      const NearChunk k = near_chunk(rp, ft, S, oa, ob);
      std::fill((uint8_t*)S.b.rec, (uint8_t*)S.seg_start, 0xA5);
      for (uint32_t i = k.n; i-- > 0;)  // any order
        if (!near_stage(rp, ft, k, i, R.view(), S)) return 1;
      S.b.z[k.n] = ~0u;
      for (uint32_t i = 1; i < k.n; ++i)
        if (S.b.z[i] < S.b.z[i - 1]) {
          std::printf("%s: staged birds out of order\n", c.name);
          return 1;
        }
      for (uint32_t o = 0; o < k.nown; ++o) {
        near_agent(rp, ft, k, st, o, S, W.view(), cnt.data(), &err, lv);
        const uint32_t gi = k.own_lo + o;
        flock_agent_global(rp, ft.step, gi, R.view(), offset.data(), V.view(), want.data(),
                           &err2, lv);
        if (!same(W.x[gi], V.x[gi]) || !same(W.y[gi], V.y[gi]) || !same(W.hx[gi], V.hx[gi]) ||
            !same(W.hy[gi], V.hy[gi])) {
          std::printf("%s: bird %u at (%a, %a): (%a, %a, %a, %a) instead of (%a, %a, %a, %a)\n",
                      c.name, R.id[gi], R.x[gi], R.y[gi], W.x[gi], W.y[gi], W.hx[gi], W.hy[gi],
                      V.x[gi], V.y[gi], V.hx[gi], V.hy[gi]);
          return 1;
        }
        ++stepped;
      }
      ++chunks;
      oa = ob;
    }
  }
  if (cnt != want || err != err2) {
    std::printf("%s: bin counts differ\n", c.name);
    return 1;
  }
  // runs of birds of one tile, staged with their neighbourhood only
  // (k_flock_runs): whole tile height across columns, else the run's rows
  uint32_t pieces = 0;
  std::vector<uint64_t> big((near_smem_bytes((int)c.n, cols) + 7) / 8 + 2);
  const NearSmem P = near_carve((uint8_t*)(((uintptr_t)big.data() + 15) & ~(uintptr_t)15),
                                (int)c.n, cols);
  for (int k = 0; k < 60; ++k) {
    uint32_t s = (uint32_t)(rng() % c.n), e = s + 1u + (uint32_t)(rng() % 200u);
    int32_t cx, cy;
    discretize(g, R.x[s], R.y[s], &cx, &cy);
    const FlockTile ft = flock_tile(&rp, 1, prefix, tile_of(g, cx, cy), 0);
    e = std::min(e, offset[ft.tb1]);
    if (k % 2) e = std::min(e, offset[rp.bin_base + col_bin0(g, ft.tile, cx & (g.tx - 1)) +
                                      (uint32_t)g.tr]);
    const int32_t ca = cell_axis(g, R.x[s]), cb = cell_axis(g, R.x[e - 1]);
    const int32_t r0 = ca == cb ? cell_axis(g, R.y[s]) : ft.y0;
    const int32_t r1 = ca == cb ? cell_axis(g, R.y[e - 1]) : ft.y1 - 1;
    const FlockTile pt = near_piece(rp, ft, ca, cb, r0, r1);
    if (pt.ncols > cols) {
      std::printf("%s: a piece of %d columns\n", c.name, pt.ncols);
      return 1;
    }
    uint32_t L = 0;
    for (int t = 0; t < pt.ncols; ++t) {
      P.col_base[t] = L;
      L += flock_segments(rp, pt, t, offset.data(), P.seg_start, P.seg_len);
    }
    P.col_base[pt.ncols] = L;
    bool ok = true;
    for (uint32_t i = 0; i < L; ++i) ok = near_stage_piece(rp, pt, i, R.view(), P) && ok;
    if (!ok) continue;
    P.b.z[L] = ~0u;
    const FlockSinks lv{Outbox{}, 0u, nullptr, nullptr, nullptr};
    for (uint32_t gi = s; gi < e; ++gi) {
      near_agent_piece(rp, pt, gi, R.view(), P, W.view(), cnt.data(), &err, lv);
      flock_agent_global(rp, ft.step, gi, R.view(), offset.data(), V.view(), want.data(), &err2,
                         lv);
      if (!same(W.x[gi], V.x[gi]) || !same(W.y[gi], V.y[gi]) || !same(W.hx[gi], V.hx[gi]) ||
          !same(W.hy[gi], V.hy[gi])) {
        std::printf("%s: bird %u of a run differs\n", c.name, R.id[gi]);
        return 1;
      }
    }
    ++pieces;
  }
  if (pieces < 10 && c.headings != 2) {
    std::printf("%s: %u runs\n", c.name, pieces);
    return 1;
  }
  std::printf("%s: %u of %u birds in %u chunks, %u tiles left to the general form\n", c.name,
              stepped, c.n, chunks, bad_tiles);
  return stepped * 4 < c.n ? 1 : 0;  // a scenario that skips most birds shows nothing
}

int main() {
  const float d = 10.0f / 1.5f;
  const float inf = INFINITY;
  const Case cases[] = {
      {"sparse", 3000, 1100, 1100, d, 10, 0.7f, 0, 0, 0, 900, 0, 0, 1, true},
      {"dense", 6000, 300, 300, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, 1, true},
      {"dense, chunked", 6000, 300, 300, d, 10, 0.7f, 8, 32, 4, 300, 0, 0, 1, true},
      {"rows for strips", 6000, 300, 300, d, 10, 0.7f, 16, 16, 1, 1400, 0, 0, 1, true},
      {"two bins to a strip", 6000, 300, 300, d, 10, 0.7f, 16, 64, 1, 3000, 0, 0, 1, true},
      {"short tiles", 2000, 400, 380, d, 10, 0.7f, 4, 4, 1, 600, 0, 0, 1, true},
      {"one-cell tiles", 800, 250, 250, d, 10, 0.7f, 1, 1, 1, 600, 0, 0, 1, true},
      {"corners", 4000, 200, 200, 5, 10, 0.7f, 0, 0, 0, 3000, 1, 0, 1, true},
      {"corners, far coordinates", 20000, 20480, 20480, d, 10, 0.7f, 16, 256, 16, 3000, 1, 0, 1,
       true},
      {"d = radius", 3000, 400, 400, 10, 10, 0.7f, 0, 0, 0, 2000, 0, 0, 1, true},
      {"d = radius, corners", 3000, 400, 400, 10, 10, 0.7f, 0, 0, 0, 3000, 1, 0, 1, true},
      {"d > radius", 3000, 400, 400, 16, 10, 0.7f, 0, 0, 0, 2000, 0, 0, 1, true},
      {"d > radius, corners", 2000, 400, 400, 16, 10, 0.7f, 0, 0, 0, 2000, 1, 0, 1, true},
      {"5 x 5 windows", 3000, 300, 300, 4, 9.5f, 0.7f, 0, 0, 0, 2500, 0, 0, 1, true},
      {"5 x 5 windows, far", 3000, 300, 300, 4, 8.0f, 0.7f, 0, 0, 0, 2500, 1, 0, 1, true},
      {"7 x 7 windows", 2000, 300, 300, 3, 10, 0.7f, 8, 32, 4, 2500, 0, 0, 1, true},
      {"crowded spot", 1500, 500, 500, d, 10, 0.7f, 8, 32, 4, 1400, 2, 0, 1, true},
      {"wide", 2000, 900, 120, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, 1, true},
      {"tall", 2000, 300, 420, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, 1, true},
      {"far edges", 2000, 300, 300, d, 10, 0.7f, 8, 8, 2, 1400, 3, 0, 1, true},
      {"far edges, whole cells", 2000, 300, 300, 10, 15, 0.7f, 8, 8, 2, 1400, 3, 0, 1, true},
      {"tiny headings", 1500, 900, 900, d, 10, 0.7f, 0, 0, 0, 900, 0, 1, 0, true},
      {"tiny headings, dense", 3000, 300, 300, d, 10, 0.7f, 0, 0, 0, 1400, 0, 1, 1, true},
      {"wild headings", 3000, 500, 500, d, 10, 0.7f, 0, 0, 0, 1400, 0, 2, 1, true},
      {"long jumps", 2000, 400, 400, d, 10, 119.0f, 0, 0, 0, 1400, 0, 0, 1, true},
      {"no jump", 2000, 400, 400, d, 10, 0.0f, 0, 0, 0, 1400, 0, 0, 1, true},
      {"negative jump and weight", 2000, 400, 400, d, 10, -3.0f, 0, 0, 0, 1400, 0, 0, -2, true},
      {"too narrow", 100, 29, 29, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, 1, false},
      {"jump across", 100, 300, 300, d, 10, 91.0f, 0, 0, 0, 1400, 0, 0, 1, false},
      {"infinite jump", 100, 300, 300, d, 10, inf, 0, 0, 0, 1400, 0, 0, 1, false},
      {"too tall", 100, 200, 310, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, 1, false},
      {"infinite weight", 100, 300, 300, d, 10, 0.7f, 0, 0, 0, 1400, 0, 0, inf, false},
      {"NaN radius", 100, 300, 300, d, NAN, 0.7f, 0, 0, 0, 1400, 0, 0, 1, false},
  };
  int failed = 0;
  for (const Case& c : cases)
    for (uint64_t seed : {1, 2, 3}) failed += run(c, seed);
  // the quotients: shared reciprocals against division
  std::mt19937_64 rng(11);
  for (uint32_t i = 0; i < 4000000u; ++i) {
    const uint32_t ub = (uint32_t)(rng() % 141 + 127 - 60) << 23 | (uint32_t)(rng() & 0x7FFFFF);
    const uint32_t ua = (uint32_t)(rng() % 120 + 127 - 60) << 23 | (uint32_t)(rng() & 0x807FFFFF);
    float a, b;
    std::memcpy(&a, &ua, 4);
    std::memcpy(&b, &ub, 4);
    if (std::fabs(a / b) >= 0x1p-126f && !same(quot(a, recip_of(b)), a / b)) ++failed;
    if (!same(quot(a, 0.1), a / 10.0f)) ++failed;
  }
  if (!same(quot(-0.0f, recip_of(3.0f)), -0.0f) || !same(quot(inf, recip_of(3.0f)), inf) ||
      !same(quot(0.0f, recip_of(0.0f)), NAN))
    ++failed;
  std::printf("%d scenario(s) failed\n", failed);
  return failed ? 1 : 0;
}
