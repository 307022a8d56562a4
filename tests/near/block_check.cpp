// block_check.cpp -- the device arrays that share an allocation (DevBlock in
// kg_common.hpp, DevBuf in kg_rt_state.hpp) over an allocator of the test's
// own: as few allocations as their sizes ask for, aligned, apart from each
// other and inside them, null when one fails or is released.  Exit status 0:
// all agree.
#define __HIP_PLATFORM_AMD__ 1
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "kg_rt_state.hpp"

static std::map<void*, size_t> live;
static int mallocs = 0;
static bool fail_next = false;
static int fail_after = -1;  // allocations that still succeed

extern "C" hipError_t hipMalloc(void** p, size_t n) {
  ++mallocs;
  *p = nullptr;
  if (fail_next || fail_after == 0) return hipErrorOutOfMemory;
  if (fail_after > 0) --fail_after;
  *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  live[*p] = n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
  if (p && !live.erase(p)) std::abort();
  std::free(p);
  return hipSuccess;
}
extern "C" hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
extern "C" hipError_t hipHostMalloc(void**, size_t, unsigned int) { return hipErrorOutOfMemory; }
extern "C" hipError_t hipHostFree(void*) { return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

using namespace kg;

#define EXPECT(c)                                                \
  do {                                                           \
    if (!(c)) {                                                  \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);        \
      return 1;                                                  \
    }                                                            \
  } while (0)

// Fills the arrays with their own bytes (the sanitizer watches the ends) and
// sees that none has another's.
static bool apart(std::initializer_list<std::pair<void*, size_t>> a) {
  uint8_t k = 0;
  for (auto& v : a) std::memset(v.first, ++k, v.second);
  k = 0;
  for (auto& v : a) {
    ++k;
    if ((uintptr_t)v.first % 256) return false;
    for (size_t i = 0; i < v.second; ++i)
      if (((uint8_t*)v.first)[i] != k) return false;
  }
  return true;
}

static int buffers(size_t cap) {
  mallocs = 0;
  DevBuf d;
  const int want = (cap + 63) / 64 * 256 < kOwnPiece ? 5 : 1;
  EXPECT(d.alloc(cap) == hipSuccess && mallocs == want && (int)live.size() == want);
  const size_t n = (cap ? cap : 1) * 4;
  EXPECT(apart({{d.b.x, n}, {d.b.y, n}, {d.b.hx, n}, {d.b.hy, n}, {d.b.id, n}}));
  d.release();
  EXPECT(live.empty() && !d.b.x && !d.b.y && !d.b.hx && !d.b.hy && !d.b.id);
  d.release();
  for (int k = 0; k < want; ++k) {
    fail_after = k;
    EXPECT(d.alloc(cap) != hipSuccess && !d.b.x && !d.b.id && live.empty());
  }
  fail_after = -1;
  d.release();
  EXPECT(live.empty());
  return 0;
}

static int blocks(size_t n, bool whole) {
  mallocs = 0;
  DevBlock b;
  uint32_t *p = nullptr, *q = nullptr;
  uint64_t* r = nullptr;
  float* s = nullptr;
  b.add(&p, n);
  b.add(&r, 3);
  b.add(&q, 0);
  b.add(&s, n + 1);
  EXPECT(b.alloc(whole) == hipSuccess && mallocs == (whole ? 1 : 4));
  EXPECT(apart({{p, n * 4}, {r, 24}, {q, 4}, {s, (n + 1) * 4}}));
  EXPECT(b.clear() == hipSuccess && (n == 0 || p[n - 1] == 0u) && r[2] == 0u && s[n] == 0.0f);
  std::swap(p, q);  // as the steps swap their offset tables
  b.release();
  EXPECT(live.empty() && !p && !q && !r && !s);
  b.add(&p, n);
  fail_next = true;
  EXPECT(b.alloc() != hipSuccess && !p);
  fail_next = false;
  b.release();
  b.add(&p, 2 * n);
  EXPECT(b.alloc() == hipSuccess && apart({{p, 8 * n}}));
  b.release();
  EXPECT(live.empty() && !p);
  return 0;
}

// n arrays of `bytes`: the allocations they take, whole or not.
static int pieces(size_t n, size_t bytes, bool whole, int want) {
  std::vector<uint8_t*> p(n);
  DevBlock b;
  for (auto& v : p) b.add(&v, bytes);
  mallocs = 0;
  EXPECT(b.alloc(whole) == hipSuccess && mallocs == want && (int)live.size() == want);
  for (size_t i = 0; i < n; ++i) std::memset(p[i], (int)i + 1, bytes);
  for (size_t i = 0; i < n; ++i)
    EXPECT((uintptr_t)p[i] % 256 == 0 && p[i][0] == i + 1 && p[i][bytes - 1] == i + 1);
  b.release();
  EXPECT(live.empty());
  for (auto& v : p) EXPECT(v == nullptr);
  // the second allocation fails: the first is given back
  if (want > 1) {
    for (auto& v : p) b.add(&v, bytes);
    fail_after = 1;
    EXPECT(b.alloc(whole) != hipSuccess && live.empty());
    fail_after = -1;
    for (auto& v : p) EXPECT(v == nullptr);
    b.release();
  }
  return 0;
}

int main() {
  int failed = 0;
  const size_t K = 1024, M = 1024 * K;
  failed += pieces(3, 60 * K, false, 3);
  failed += pieces(30, 590 * K, false, 30);       // small: pieces of their own
  failed += pieces(30, 590 * K, true, 1);         // little else allocated
  failed += pieces(30, M, false, 30);             // one to a block
  failed += pieces(8, M + 512 * K, false, 8);
  failed += pieces(64, M, false, 64);             // the largest split
  failed += pieces(65, M, false, 1);
  failed += pieces(5, 2 * M, false, 1);           // past the runtime's block
  failed += pieces(1, 0 + 5 * M, false, 1);
  for (size_t n : {0, 1, 63, 64, 65, 1000, 4096, 262080, 262081, 300000})
    failed += buffers(n) + blocks(n % 5000, false) + blocks(n % 5000, true);
  std::printf("%d scenario(s) failed\n", failed);
  return failed ? 1 : 0;
}
