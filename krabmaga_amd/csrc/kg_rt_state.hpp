// kg_rt_state.hpp -- device memory of the tile-resident layout (kg_rt.hpp)
// and the host mirror of its step counter, shared by the plain field and
// the ensemble engine.
#pragma once

#include "kg_common.hpp"

namespace kg {

// An agent buffer, its five arrays apart (small ones) or in one allocation,
// that of x; or part of a block that owns them.
struct DevBuf {
  Buf b{};
  bool apart = false;
  hipError_t alloc(size_t cap) {
    const size_t stride = ((cap ? cap : 1) + 63) / 64 * 64;  // 256 bytes
    b = Buf{};
    apart = stride * sizeof(float) < kOwnPiece;
    hipError_t e;
    if (apart) {
      if ((e = dmalloc(&b.x, stride)) != hipSuccess || (e = dmalloc(&b.y, stride)) != hipSuccess ||
          (e = dmalloc(&b.hx, stride)) != hipSuccess ||
          (e = dmalloc(&b.hy, stride)) != hipSuccess || (e = dmalloc(&b.id, stride)) != hipSuccess)
        release();
      return e;
    }
    float* p = nullptr;
    if ((e = dmalloc(&p, 5 * stride)) == hipSuccess)
      b = Buf{p, p + stride, p + 2 * stride, p + 3 * stride, (uint32_t*)(p + 4 * stride)};
    return e;
  }
  void release() {
    if (apart)
      for (void* p : {(void*)b.y, (void*)b.hx, (void*)b.hy, (void*)b.id}) (void)hipFree(p);
    (void)hipFree(b.x);
    b = Buf{};
  }
};

inline void add_buf(DevBlock* block, Buf* b, size_t cap) {
  block->add(&b->x, cap);
  block->add(&b->y, cap);
  block->add(&b->hx, cap);
  block->add(&b->hy, cap);
  block->add(&b->id, cap);
}

struct RtState {
  bool allocated = false;
  RtPlan plan;
  int ncls = 2;
  RtCaps caps[kRtMaxClasses]{};
  uint32_t* dense = nullptr;  // device tile lists of classes 1.., grouped by class
  uint32_t off[kRtMaxClasses + 1] = {};
  uint32_t ndense = 0;
  std::vector<uint32_t> dense_host;  // kept until the upload ran
  uint32_t ntiles = 0;
  uint64_t stay_alloc = 0, inbox_alloc = 0, boff_alloc = 0, spill_alloc = 0, tiles_alloc = 0;
  RtMeta* meta = nullptr;  // per tile
  uint32_t *cnt[2] = {nullptr, nullptr}, *boff[2] = {nullptr, nullptr};
  uint32_t* icnt[3] = {nullptr, nullptr, nullptr};
  uint32_t* scnt = nullptr;  // 3 counters
  Buf stay[2]{}, inbox[2]{}, spill[2]{};
  Buf out{};  // unload target (if asked for), of the spill lists' capacity
  uint32_t* spill_rep[2] = {nullptr, nullptr};
  uint32_t* flags = nullptr;
  uint64_t* gstep = nullptr;
  uint32_t* ovf = nullptr;  // 2 x (kRtOvfMax + 1)
  DevBlock block;  // every device array above
  uint64_t G = 0;  // value of *gstep once queued work has run
  std::vector<std::pair<int, hipGraphExec_t>> graphs;  // (steps, exec)
  // the class launches of a step run side by side on these streams
  hipStream_t aux[kRtMaxClasses] = {};
  hipEvent_t ev_fork = nullptr, ev_done[kRtMaxClasses] = {};

  RtDev dev() const;
  // (Re)allocates for `plan` (growing only), with room for spill_cap agents
  // in each spill list and in `out` (with_out), and uploads the plan tables
  // and the class split.
  int setup(const RtPlan& plan, const RtClassPlan& cls, uint64_t spill_cap, hipStream_t s,
            bool with_out = false);
  // Zeroes the counters and flags and sets the step counter to G.
  int reset(uint64_t G, hipStream_t s);
  void drop_graphs();
  void release();
};

hipError_t launch_set_u64(uint64_t* p, uint64_t v, hipStream_t s);

// One tile-resident schedule step, launch koff of a batch: the class
// launches of the plan in `rt` side by side (they touch disjoint tiles), then
// one launch for the tiles they deferred.
hipError_t rt_launch_classes(const WorkList& wl, const RtDev& D, const RtState& rt, uint32_t koff,
                             hipStream_t s);
hipError_t launch_add_u64(uint64_t* p, uint64_t v, hipStream_t s);

}  // namespace kg
