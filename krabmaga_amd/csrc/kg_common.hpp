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

// Device arrays that live and die together, in as many allocations as pay.
// What one costs depends on what else is allocated and freed (MI355X, ROCm
// 7.2).  Arrays under 1 MiB or so come out of 2 MiB blocks that the runtime
// keeps while something is left in them, about 1 us each.  Larger ones are
// mapped anew, 12 us, but once eight or so have been freed in a row the frees
// are put off and whatever allocates next (a stream, a graph) waits 0.2 to 1.2
// ms.  So arrays are allocated apart while all of them are small, then in
// pieces of the runtime's block size up to a total of 64 MiB, then in one
// piece; and in one piece where the object has little else (`whole`).
// Ensembles admitted, run, read and closed, ms, every array apart and so: 12
// runs up to 120,000 birds, 60 steps, 16.7 and 8.5; 50 up to 30,000, 100 steps,
// 31.0 and 18.3; 30 up to 5,000, served, 9.8 and 9.7 (10.2 in one piece).
constexpr size_t kOwnPiece = 1u << 20;  // smaller arrays are allocated by themselves

class DevBlock {
 public:
  // n elements for *p, from the next alloc() on; p stays valid till release().
  template <class T>
  void add(T** p, size_t n) {
    parts_.push_back({p, ((n ? n : 1) * sizeof(T) + kAlign - 1) / kAlign * kAlign, 0, 0});
  }
  hipError_t alloc(bool whole = false) {
    size_t total = 0, largest = 0;
    for (const Part& q : parts_) {
      total += q.size;
      largest = q.size > largest ? q.size : largest;
    }
    size_t cut = total;  // bytes of a piece, at most, or those of one array
    if (!whole && largest < kOwnPiece) cut = 0;
    else if (!whole && largest <= kPiece && total <= kSplit) cut = kPiece;
    for (Part& q : parts_) {
      if (pieces_.empty() || pieces_.back().size + q.size > cut) pieces_.push_back({nullptr, 0});
      q.piece = pieces_.size() - 1;
      q.at = pieces_.back().size;
      pieces_.back().size += q.size;
    }
    hipError_t e = hipSuccess;
    for (Piece& q : pieces_)
      if (e == hipSuccess && (e = hipMalloc(&q.base, q.size)) != hipSuccess) q.base = nullptr;
    if (e != hipSuccess) free_pieces();
    set();
    return e;
  }
  // Every array to zero (not for a captured graph).
  hipError_t clear() {
    hipError_t e = hipSuccess;
    for (const Piece& q : pieces_)
      if (e == hipSuccess) e = hipMemset(q.base, 0, q.size);
    return e;
  }
  void release() {
    free_pieces();
    set();
    parts_.clear();
    pieces_.clear();
  }

 private:
  struct Piece {
    void* base;
    size_t size;
  };
  struct Part {
    void* p;  // where the array's pointer is
    size_t size;
    size_t piece, at;
  };
  static constexpr size_t kAlign = 256;
  static constexpr size_t kPiece = (2u << 20) - (64u << 10), kSplit = 64u << 20;
  void free_pieces() {
    for (Piece& q : pieces_) {
      if (q.base) (void)hipFree(q.base);
      q.base = nullptr;
    }
  }
  void set() {
    for (const Part& q : parts_) {
      void* const b = pieces_.empty() ? nullptr : pieces_[q.piece].base;
      void* const v = b ? (uint8_t*)b + q.at : nullptr;
      std::memcpy(q.p, &v, sizeof(v));  // a pointer of the array's own type
    }
  }
  std::vector<Part> parts_;
  std::vector<Piece> pieces_;
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
