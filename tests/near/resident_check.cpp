// resident_check.cpp -- the resident step's phases (kg_resident.hpp) on the
// CPU against the general form on the read buffer's layout, bit for bit over
// several steps, with the final order of the read buffer.  Exit status 0:
// every scenario agrees.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "kg_geom.hpp"
#include "kg_resident.hpp"

using namespace kg;

struct Case {
  const char* name;
  uint32_t n;
  float w, h, d, radius, jump;
  uint32_t tx, ty, hb;
  uint32_t bins;  // bin table (0: res_fits' own); small ones give tall bins
  int layout;     // 0 uniform, 1 one crowded spot, 2 some outside [0, w]
  uint32_t steps;
};

struct Cols {
  std::vector<float> x, y, hx, hy;
  std::vector<uint32_t> id;
  explicit Cols(size_t n) : x(n), y(n), hx(n), hy(n), id(n) {}
  Buf view() { return Buf{x.data(), y.data(), hx.data(), hy.data(), id.data()}; }
};

// The read buffer of `A`: (bin, row, id) order and the bin offsets.
static void sort_api(const Geom& g, const Cols& A, Cols* R, std::vector<uint32_t>* offset) {
  const uint32_t n = (uint32_t)A.x.size();
  std::vector<uint32_t> ord(n), bin(n);
  std::vector<int32_t> row(n);
  offset->assign(g.nbins + 1, 0u);
  for (uint32_t i = 0; i < n; ++i) {
    int32_t cx;
    discretize(g, A.x[i], A.y[i], &cx, &row[i]);
    bin[i] = bin_of(g, cx, row[i]);
    ++(*offset)[bin[i] + 1];
    ord[i] = i;
  }
  for (uint32_t b = 0; b < g.nbins; ++b) (*offset)[b + 1] += (*offset)[b];
  std::sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) {
    if (bin[a] != bin[b]) return bin[a] < bin[b];
    if (row[a] != row[b]) return row[a] < row[b];
    return A.id[a] < A.id[b];
  });
  for (uint32_t k = 0; k < n; ++k) {
    R->x[k] = A.x[ord[k]];
    R->y[k] = A.y[ord[k]];
    R->hx[k] = A.hx[ord[k]];
    R->hy[k] = A.hy[ord[k]];
    R->id[k] = A.id[ord[k]];
  }
}

static int run(const Case& c, uint64_t seed) {
  Geom g{};
  std::string why;
  if (!make_geom_rt(c.w, c.h, c.d, 1, c.n, c.tx, c.ty, c.hb, &g, &why, true)) {
    std::printf("%s: %s\n", c.name, why.c_str());
    return 1;
  }
  RepDev rp{};
  rp.g = g;
  kg_flock_params p{1.2f, 0.8f, 1.3f, 0.7f, 0.9f, c.jump, c.radius, 0u, seed};
  set_rep_params(&rp, p);
  uint32_t bins = 0;
  if (!res_fits(rp, c.n, 157696, &bins)) {
    std::printf("%s: does not fit\n", c.name);
    return 1;
  }
  if (c.bins) bins = std::max<uint32_t>({c.bins, (uint32_t)g.dw, g.nbins});
  std::mt19937_64 rng(seed * 104729 + c.n);
  auto u = [&] { return (float)(rng() >> 40) * 0x1p-24f; };
  Cols A(c.n), R(c.n), W(c.n);
  for (uint32_t i = 0; i < c.n; ++i) {
    A.x[i] = c.w * u();
    A.y[i] = c.h * u();
    if (c.layout == 1 && i % 3) {
      A.x[i] = c.w * 0.5f + 8.0f * u();
      A.y[i] = c.h * 0.25f + 8.0f * u();
    }
    if (c.layout == 2 && i % 50 == 0) A.x[i] = c.w + 0.5f * u();
    int32_t cx, cy;
    discretize(g, A.x[i], A.y[i], &cx, &cy);
    if (!cell_valid(g, cx, cy)) A.x[i] = 1.0f;
    const float a = 6.2831853f * u();
    A.hx[i] = std::cos(a);
    A.hy[i] = std::sin(a);
    A.id[i] = i;
  }
  std::vector<uint32_t> offset;
  sort_api(g, A, &R, &offset);
  // the resident run
  std::vector<uint64_t> smem((res_smem_bytes(c.n, bins) + 7) / 8 + 2);
  const ResSmem S = res_carve((uint8_t*)(((uintptr_t)smem.data() + 15) & ~(uintptr_t)15), c.n);
  const ResBins rb = res_bins(g, bins);
  const CellFind find{S.b.z, S.tab, rb.rows, rb.shift};
  std::vector<ResBird> b(c.n);
  for (uint32_t i = 0; i < c.n; ++i)
    b[i] = ResBird{R.x[i], R.y[i], R.hx[i], R.hy[i], R.id[i], 0u, 0u, 0u};
  uint32_t err = 0, general = 0;
  for (uint32_t k = 0;; ++k) {
    const bool last = k == c.steps;
    const uint32_t nb = last ? g.nbins : rb.n;
    if (nb > bins) return 1;
    std::fill(S.tab, S.tab + nb, 0u);
    bool bad = !rp.near;
    for (uint32_t i : [&] {  // any order of the counting
           std::vector<uint32_t> o(c.n);
           for (uint32_t q = 0; q < c.n; ++q) o[q] = q;
           std::shuffle(o.begin(), o.end(), rng);
           return o;
         }()) {
      res_place(rp, rb, last, &b[i], &err);
      b[i].slot = S.tab[b[i].bin]++;
      if (near_bad(g, b[i].x, b[i].y, b[i].hx, b[i].hy)) bad = true;
    }
    uint32_t run = 0;
    for (uint32_t q = 0; q < nb; ++q) {
      const uint32_t v = S.tab[q];
      S.tab[q] = run;
      run += v;
    }
    S.tab[nb] = run;
    uint64_t* key = (uint64_t*)S.b.rec;
    for (auto& q : b) key[S.tab[q.bin] + q.slot] = res_key(q);
    for (auto& q : b)
      q.slot = S.tab[q.bin] + gather_rank(key, S.tab[q.bin], S.tab[q.bin + 1],
                                          S.tab[q.bin] + q.slot, res_key(q));
    if (last) break;
    for (auto& q : b) {
      S.b.rec[q.slot] = NearRec{q.x, q.y, q.hx, q.hy};
      S.b.z[q.slot] = q.z;
      S.b.id[q.slot] = q.id;
    }
    S.b.z[c.n] = ~0u;
    general += bad;
    // the general form on the read buffer
    std::vector<uint32_t> cnt(g.nbins, 0u);
    rp.step_base = k;
    for (uint32_t i = 0; i < c.n; ++i)
      flock_agent_global(rp, k, i, R.view(), offset.data(), W.view(), cnt.data(), &err,
                         FlockSinks{Outbox{}, 0u, nullptr, nullptr, nullptr});
    W.id = R.id;
    std::vector<uint32_t> at(c.n);
    for (uint32_t i = 0; i < c.n; ++i) at[W.id[i]] = i;
    for (uint32_t i = 0; i < c.n; ++i) {
      ResBird& q = b[i];
      NearRec r;
      if (bad) full_step(rp, k, i, find, S.b, &r);
      else near_step<true>(rp, 0, k, i, find, S.b, &r);
      q.x = r.x;
      q.y = r.y;
      q.hx = r.hx;
      q.hy = r.hy;
      q.id = S.b.id[i];
      const uint32_t j = at[q.id];
      if (std::memcmp(&q.x, &W.x[j], 4) || std::memcmp(&q.y, &W.y[j], 4) ||
          std::memcmp(&q.hx, &W.hx[j], 4) || std::memcmp(&q.hy, &W.hy[j], 4)) {
        std::printf("%s: step %u bird %u: (%a, %a) instead of (%a, %a)\n", c.name, k, q.id, q.x,
                    q.y, W.x[j], W.y[j]);
        return 1;
      }
    }
    Cols next = W;
    sort_api(g, next, &R, &offset);
  }
  for (uint32_t q = 0; q < g.nbins; ++q)
    if (S.tab[q] != offset[q]) {
      std::printf("%s: bin offsets differ\n", c.name);
      return 1;
    }
  for (auto& q : b)
    if (R.id[q.slot] != q.id) {
      std::printf("%s: order differs\n", c.name);
      return 1;
    }
  std::printf("%s: %u birds, %u steps, shift %d, %u steps in the general form\n", c.name, c.n,
              c.steps, rb.shift, general);
  return err ? 1 : 0;
}

int main() {
  const float d = 10.0f / 1.5f;
  const Case cases[] = {
      {"one bird", 1, 200, 200, d, 10, 0.7f, 0, 0, 0, 0, 0, 4},
      {"two birds", 2, 60, 60, d, 10, 0.7f, 0, 0, 0, 0, 0, 30},
      {"1,000 boids", 1000, 200, 200, d, 10, 0.7f, 0, 0, 0, 0, 0, 12},
      {"tall bins", 1000, 200, 200, d, 10, 0.7f, 8, 32, 16, 40, 0, 6},
      {"sparse", 1500, 774, 774, d, 10, 0.7f, 0, 0, 0, 0, 0, 8},
      {"very sparse", 300, 3000, 3000, d, 10, 0.7f, 32, 256, 64, 0, 0, 3},
      {"full", 4096, 404.8f, 404.8f, d, 10, 0.7f, 0, 0, 0, 0, 0, 3},
      {"crowded spot", 900, 300, 300, d, 10, 0.7f, 0, 0, 0, 0, 1, 5},
      {"tall", 600, 100, 140, d, 10, 0.7f, 0, 0, 0, 0, 0, 6},
      {"outside the width", 900, 199, 199, d, 10, 0.7f, 0, 0, 0, 0, 2, 4},
      {"narrow torus", 40, 25, 25, d, 10, 0.7f, 0, 0, 0, 0, 0, 8},
      {"one cell", 30, 5, 5, d, 10, 0.7f, 0, 0, 0, 0, 0, 4},
      {"long jumps", 500, 200, 200, d, 10, 150.0f, 0, 0, 0, 0, 0, 5},
      {"5 x 5 windows", 800, 200, 200, 4, 9.5f, 0.7f, 0, 0, 0, 0, 0, 5},
      {"d > radius", 800, 300, 300, 16, 10, 0.7f, 0, 0, 0, 0, 0, 5},
      {"tiles of 4 x 4", 800, 300, 300, d, 10, 0.7f, 4, 4, 2, 0, 0, 5},
  };
  int failed = 0;
  for (const Case& c : cases)
    for (uint64_t seed : {1, 2}) failed += run(c, seed);
  std::printf("%d scenario(s) failed\n", failed);
  return failed ? 1 : 0;
}
