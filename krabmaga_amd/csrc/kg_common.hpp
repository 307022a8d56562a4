// kg_common.hpp -- host-side helpers shared by the C ABI implementations.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/krabgpu.h"
#include "kg_geom.hpp"
#include "kg_launch.hpp"

namespace kg {

// Records the message of the failing call for kg_last_error (per thread).
int set_error(int code, const char* fmt, ...);
void clear_error();

// Largest flock-kernel LDS capacity (staged agents) at or below `cap` whose
// dynamic plus static LDS fits the device's per-block limit.
int clamp_lds_cap(int cap);

// The near flock kernel's staging for tiles of `cols` columns expected to
// stage `cap` birds (pick_lds_cap), `ntiles` work-groups in the launch; full:
// as near_threads.
NearPlan near_plan(int cap, int cols, uint32_t ntiles, bool full);

// Three-kernel steps per captured graph in a run of n: the GPU idles about
// 8 us between graph launches, 4 us per step with two steps to a graph
// (of 28 at 16,384 boids), while a graph of sixteen takes its capture and
// instantiation before the first launch.  Even, so that the buffers are back
// in place.
inline int graph_steps(uint32_t n) { return n >= 64u ? 16 : 2; }

// The gather rebinning after flock steps; KG_REBIN_GATHER=0 turns it off
// (scatter and bin sort every step), for comparison.
bool rebin_gather_enabled();

#define KG_HIP(expr)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess)                                                              \
      return ::kg::set_error(KG_E_HIP, "%s failed: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

template <class T>
hipError_t dmalloc(T** p, size_t n) {
  return hipMalloc((void**)p, (n ? n : 1) * sizeof(T));
}

// Device arrays that live and die together, in one allocation.  hipFree puts
// off the release of more than about eight blocks at a time, and each
// hipMalloc after that waits 200 us for one of them (MI355X, blocks past
// 2 MiB).  An ensemble of 12 runs and 60 steps, admitted, run, read and closed:
// 16.7 ms with its 75 arrays apart, 8.3 ms with them in eight blocks.
class DevBlock {
 public:
  // n elements for *p, from the next alloc() on; p stays valid till release().
  template <class T>
  void add(T** p, size_t n) {
    parts_.push_back({p, size_});
    size_ += ((n ? n : 1) * sizeof(T) + kAlign - 1) / kAlign * kAlign;
  }
  hipError_t alloc() {
    const hipError_t e = hipMalloc(&base_, size_ ? size_ : kAlign);
    if (e != hipSuccess) base_ = nullptr;
    set();
    return e;
  }
  // Every array to zero (not for a captured graph).
  hipError_t clear() { return hipMemset(base_, 0, size_); }
  void release() {
    if (base_) (void)hipFree(base_);
    base_ = nullptr;
    set();
    parts_.clear();
    size_ = 0;
  }

 private:
  static constexpr size_t kAlign = 256;
  void set() {
    for (const auto& q : parts_) {
      void* const v = base_ ? (uint8_t*)base_ + q.second : nullptr;
      std::memcpy(q.first, &v, sizeof(v));  // a pointer of the array's own type
    }
  }
  std::vector<std::pair<void*, size_t>> parts_;  // where the array's pointer is, its offset
  void* base_ = nullptr;
  size_t size_ = 0;
};

// Pinned host memory of one object for reading small buffers (launch_pack),
// allocated at the first read and given back with the object.  Larger buffers
// are copied straight to the caller (past about 32,000 agents the copies'
// bandwidth outweighs their calls).
constexpr size_t kStageAgents = 32768;

struct HostStage {
  uint32_t* p = nullptr;
  size_t words = 0;

  static bool fits(size_t n) { return n <= kStageAgents; }
  // Room for n agents (fits(n)); false if the allocation fails.
  bool reserve(size_t n) {
    const size_t want = kPackHead + 5 * n;
    if (want <= words) return true;
    release();
    if (hipHostMalloc((void**)&p, want * sizeof(uint32_t)) != hipSuccess) {
      p = nullptr;
      (void)hipGetLastError();
      return false;
    }
    words = want;
    return true;
  }
  // The n packed agents to the caller's arrays (any may be null).
  void unpack(size_t n, uint32_t* ids, float* x, float* y, float* hx, float* hy) const {
    void* const dst[5] = {x, y, hx, hy, ids};
    for (size_t k = 0; k < 5; ++k)
      if (dst[k] && n) std::memcpy(dst[k], p + kPackHead + k * n, n * sizeof(uint32_t));
  }
  void release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    words = 0;
  }
};

}  // namespace kg
