// gather_check.cpp -- the slow way of the gather rebinning (kg_phases.hpp) on
// the CPU, tile by tile as the kernel takes it: outboxes that overflowed read
// as whole tiles, birds from further than the neighbours found in the whole
// replica, bins sorted in place by the bitonic network.  The result is the
// (bin, row, id) order of all birds.  Exit status 0: every scenario agrees.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <random>
#include <vector>

#include "kg_geom.hpp"
#include "kg_phases.hpp"

using namespace kg;

struct Cols {
  std::vector<float> x, y, hx, hy;
  std::vector<uint32_t> id;
  explicit Cols(size_t n) : x(n), y(n), hx(n), hy(n), id(n) {}
  Buf view() { return Buf{x.data(), y.data(), hx.data(), hy.data(), id.data()}; }
};

struct Case {
  const char* name;
  uint32_t n, crowd;  // birds, those of them in one cell
  float side, jump;
  uint32_t far;  // birds whose position becomes NaN
  uint32_t tx, ty, hb;
};

static uint32_t bin_at(const Geom& g, float x, float y, int32_t* row) {
  *row = cell_axis(g, y);
  return bin_of(g, cell_axis(g, x), *row);
}

// Order of v's birds by (bin, row, id), and the bins' starts.
static std::vector<uint32_t> order_of(const Geom& g, const Cols& v, std::vector<uint32_t>* offset) {
  const uint32_t n = (uint32_t)v.x.size();
  std::vector<uint32_t> ord(n), bin(n);
  std::vector<int32_t> row(n);
  offset->assign(g.nbins + 1, 0u);
  for (uint32_t i = 0; i < n; ++i) ++(*offset)[(bin[i] = bin_at(g, v.x[i], v.y[i], &row[i])) + 1];
  std::partial_sum(offset->begin(), offset->end(), offset->begin());
  std::iota(ord.begin(), ord.end(), 0u);
  std::sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) {
    if (bin[a] != bin[b]) return bin[a] < bin[b];
    if (row[a] != row[b]) return row[a] < row[b];
    return v.id[a] < v.id[b];
  });
  return ord;
}

static int run(const Case& c, uint64_t seed) {
  RepDev rp{};
  std::string why;
  if (!make_geom_rt(c.side, c.side, 10.0f / 1.5f, 1, c.n, c.tx, c.ty, c.hb, &rp.g, &why)) {
    std::printf("%s: %s\n", c.name, why.c_str());
    return 1;
  }
  const Geom& g = rp.g;
  const uint32_t nbt = 1u << (g.tx_log2 + g.tr_log2);
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<float> U(0.0f, 1.0f);
  // the read buffer in order, then a step of every bird
  Cols A(c.n), R(c.n), W(c.n), R2(c.n);
  for (uint32_t i = 0; i < c.n; ++i) {
    A.x[i] = i < c.crowd ? (2.05f + 0.9f * U(rng)) * g.d : U(rng) * c.side * 0.9999f;
    A.y[i] = i < c.crowd ? (3.05f + 0.9f * U(rng)) * g.d : U(rng) * c.side * 0.9999f;
    A.id[i] = i;
  }
  std::shuffle(A.id.begin(), A.id.end(), rng);
  std::vector<uint32_t> off, off2;
  std::vector<uint32_t> ord = order_of(g, A, &off);
  for (uint32_t i = 0; i < c.n; ++i) {
    const uint32_t k = ord[i];
    R.x[i] = A.x[k];
    R.y[i] = A.y[k];
    R.id[i] = W.id[i] = A.id[k];
    const float a = 6.2831f * U(rng);
    auto wrap = [&](float v) { return v >= c.side ? v - c.side : (v < 0.0f ? v + c.side : v); };
    W.x[i] = wrap(R.x[i] + c.jump * std::cos(a));
    W.y[i] = wrap(R.y[i] + c.jump * std::sin(a));
    W.hx[i] = U(rng);
    W.hy[i] = U(rng);
  }
  for (uint32_t k = 0; k < c.far; ++k) W.x[rng() % c.n] = NAN;
  for (uint32_t k = 0; k < c.far; ++k) W.y[rng() % c.n] = NAN;
  ord = order_of(g, W, &off2);
  // the outboxes: a tile's leavers, the first kOutboxCap of them listed
  std::vector<uint32_t> on(g.ntiles, 0u), slot((size_t)g.ntiles * kOutboxCap, 0u);
  for (uint32_t tile = 0; tile < g.ntiles; ++tile)
    for (uint32_t i = off[tile * nbt]; i < off[(tile + 1) * nbt]; ++i) {
      int32_t row;
      if (bin_at(g, W.x[i], W.y[i], &row) / nbt == tile) continue;
      if (on[tile] < kOutboxCap) slot[(size_t)tile * kOutboxCap + on[tile]] = i;
      ++on[tile];
    }
  const Outbox ob{on.data(), slot.data()};
  const Buf r = R.view(), w = W.view(), r2 = R2.view();
  uint32_t over = 0, whole_tiles = 0, big = 0;
  for (uint32_t v : on) over += v > kOutboxCap;
  for (uint32_t tile = 0; tile < g.ntiles; ++tile) {
    const uint32_t nlo = off2[tile * nbt], lo = off[tile * nbt], nown = off[(tile + 1) * nbt] - lo;
    std::vector<uint32_t> bstart(nbt + 1), fill(nbt), sitem(kGatherSources), scnt(kGatherSources);
    for (uint32_t b = 0; b <= nbt; ++b) bstart[b] = off2[tile * nbt + b] - nlo;
    for (uint32_t q = 0; q < kGatherSources; ++q) {
      const int32_t sl = gather_source(g, tile, q);
      sitem[q] = sl >= 0 ? (uint32_t)sl : 0u;
      scnt[q] = sl >= 0 ? on[sl] : 0u;
    }
    auto take = [&](const uint32_t* list, uint32_t base, uint32_t n) {
      for (uint32_t i = 0; i < n; ++i)
        gather_take(g, tile, nlo, bstart.data(), fill.data(), r, w, list ? list[i] : base + i, r2);
    };
    bool full = false;
    for (int whole = 0; whole < 2 && !full; ++whole) {
      std::fill(fill.begin(), fill.end(), 0u);
      if (whole) {
        ++whole_tiles;
        take(nullptr, off[0], off[g.nbins] - off[0]);
      } else {
        take(nullptr, lo, nown);
        gather_slow_sources(ob, sitem.data(), scnt.data(), off.data(), 0u, 0u, nbt, take);
      }
      full = true;
      for (uint32_t b = 0; b < nbt; ++b) full = full && fill[b] == bstart[b + 1] - bstart[b];
    }
    if (!full) {
      std::printf("%s: tile %u is short of birds\n", c.name, tile);
      return 1;
    }
    for (uint32_t b = 0; b < nbt; ++b) {
      const uint32_t m = bstart[b + 1] - bstart[b];
      big = std::max(big, m);
      bitonic_passes(m, [&](uint32_t x) {
        for (uint32_t i = 0; i < m; ++i)
          if ((i ^ x) > i && (i ^ x) < m) sort_exchange(g, r2, nlo + bstart[b], i, i ^ x);
      });
    }
  }
  for (uint32_t k = 0; k < c.n; ++k)
    if (R2.id[k] != W.id[ord[k]] || std::memcmp(&R2.x[k], &W.x[ord[k]], 4) ||
        std::memcmp(&R2.y[k], &W.y[ord[k]], 4) || R2.hx[k] != W.hx[ord[k]] ||
        R2.hy[k] != W.hy[ord[k]]) {
      std::printf("%s: slot %u holds bird %u instead of %u\n", c.name, k, R2.id[k], W.id[ord[k]]);
      return 1;
    }
  std::printf("%s: %u tiles, %u outboxes overflowed, %u tiles from the whole replica, largest bin "
              "%u\n", c.name, g.ntiles, over, whole_tiles, big);
  if (c.jump > 40.0f && over == 0) return 1;
  // (every tile neighbours cell 0 on a small grid)
  if (c.far && g.ntiles > 9 && whole_tiles == 0) return 1;
  return 0;
}

int main() {
  const Case cases[] = {
      {"steps of a cell", 6000, 0, 400, 0.7f, 0, 0, 0, 0},
      {"overflowing outboxes", 16000, 0, 400, 50.0f, 0, 8, 32, 1},
      {"birds without a position", 6000, 0, 700, 0.7f, 6, 0, 0, 0},
      {"a bin of 3,000", 5000, 3000, 400, 0.05f, 0, 0, 0, 0},
      {"a bin of 2,049", 4000, 2049, 400, 0.01f, 0, 0, 0, 0},
      {"crowd and jumps", 9000, 5000, 400, 50.0f, 3, 8, 32, 4},
      {"two tiles across", 3000, 0, 100, 0.7f, 0, 8, 8, 1},
      {"one tile", 500, 0, 40, 0.7f, 2, 0, 0, 0},
  };
  int failed = 0;
  for (const Case& c : cases)
    for (uint64_t seed : {1, 2}) failed += run(c, seed);
  // the network alone, at every small size and around powers of two
  Geom g{};
  std::string why;
  make_geom_rt(400, 400, 10.0f / 1.5f, 1, 1000, 0, 0, 0, &g, &why);
  std::mt19937 rng(3);
  for (uint32_t m : {0, 1, 2, 3, 5, 7, 8, 9, 31, 33, 255, 256, 257, 1000, 2047, 2048, 2049, 4097}) {
    Cols v(m);
    for (uint32_t i = 0; i < m; ++i) {
      v.y[i] = (float)(rng() % 100);
      v.id[i] = rng() % 50;  // ties too
    }
    bitonic_passes(m, [&](uint32_t x) {
      for (uint32_t i = 0; i < m; ++i)
        if ((i ^ x) > i && (i ^ x) < m) sort_exchange(g, v.view(), 0u, i, i ^ x);
    });
    for (uint32_t i = 1; i < m; ++i)
      if (bin_key(g, v.y[i], v.id[i]) < bin_key(g, v.y[i - 1], v.id[i - 1])) {
        std::printf("network of %u: out of order\n", m);
        ++failed;
        break;
      }
  }
  std::printf("%d scenario(s) failed\n", failed);
  return failed ? 1 : 0;
}
