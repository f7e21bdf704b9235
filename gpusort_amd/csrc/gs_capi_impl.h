// Shared host state behind the C ABI: the handle, its HBM arena, the error
// channel and the device scope guard.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/gpusort_hip.h"
#include "gs_internal.h"
#include "pinned_stage.h"

namespace gs {

// Event-pair timing of kernel launches (gs_profile_begin / gs_profile_end).
class Profiler : public LaunchTimer {
 public:
  struct Rec {
    std::string name;
    uint64_t bytes;
    hipEvent_t start, stop;
    const SortCtrl* watched;  // pinned, filled before `start`; null: it counts
    int pass;
    // Whether the launch did its work (once its stop event has passed).
    bool ran() const {
      if (!watched) return true;
      if (pass == kTiePass) return watched->low() != 0;
      return watched->src[pass] == kSkipPass ? false
             : watched->src[pass] & kCopyPass ? true
                                              : (uint32_t)pass >= watched->low();
    }
  };
  ~Profiler() override;
  void begin(const char* name, uint64_t bytes, hipStream_t stream) override;
  void end(hipStream_t stream) override;
  const SortCtrl* watch(const SortCtrl* d_ctrl, hipStream_t stream) override;
  void only_if(const SortCtrl* watched, int pass) override;
  void reset();
  std::vector<Rec> recs;
  bool active = false;

 private:
  static constexpr size_t kWatchBlock = 128;
  std::vector<hipEvent_t> pool_;
  size_t used_ = 0;
  std::vector<SortCtrl*> watch_pool_;  // pinned, kWatchBlock each
  size_t watch_used_ = 0;
  hipEvent_t take();
};

// Grow-only device buffers, one per use.  A slot is reallocated only when a
// call needs more bytes than it holds (after the stream drains); steady-state
// calls of a given size therefore allocate nothing.
class Arena {
 public:
  enum Slot { kRadix = 0, kStageKeys, kStageVals, kStagePairs, kMerge, kSmall, kPipeKeys, kPipeVals, kPipeAux,
              kSegAux, kSegWork, kHykWork, kGather, kSlots };
  Arena() {
    for (int i = 0; i < kSlots; ++i) {
      ptr_[i] = nullptr;
      cap_[i] = 0;
    }
  }
  ~Arena();
  hipError_t get(int slot, size_t bytes, hipStream_t stream, void** out);
  // hipMalloc for what a call cannot do without: where there is no memory left,
  // the gather's scratch, which the gather can do without, is given back first.
  hipError_t allocate(void** out, size_t bytes);
  // Bytes a slot allocates when it must grow to hold `bytes` (1/8 headroom,
  // whole MiB).
  static size_t grown(size_t bytes) {
    if (bytes == 0) bytes = 256;
    const size_t b = bytes + bytes / 8;
    return (b + (1u << 20) - 1) & ~(size_t)((1u << 20) - 1);
  }
  size_t bytes() const;
  void release();

  // The gather's scratch: gathers from several threads queue one after
  // another, and one on another stream than the last waits for it.
  std::mutex gather_mutex;
  hipEvent_t gather_done = nullptr;
  hipStream_t gather_stream = nullptr;

 private:
  void* ptr_[kSlots];
  size_t cap_[kSlots];
};

// Pinned host memory for the small transfers of a call (plans and offset
// tables up, samples and bounds down): copies through it return at once, where
// one from pageable memory takes 10-20 us of the host's time and the wait that
// its source needs.  Handed out front to back; when it is used up the stream is
// drained and it starts over.
class PinnedStage {
 public:
  static constexpr size_t kBytes = 4u << 20;
  // Room for `bytes`, or null (too large, or no pinned memory): the caller then
  // copies from and to its own memory.  Good until the next call may start over:
  // blocks that are read together take one room (read_staged).
  void* take(size_t bytes, hipStream_t stream);
  void release();

 private:
  char* base_ = nullptr;
  StageRing ring_{kBytes};
  bool failed_ = false;
};

class DeviceScope {
 public:
  explicit DeviceScope(int dev);
  ~DeviceScope();

 private:
  int prev_ = -1;
  int dev_ = 0;
};

gs_status fail(gs_status st, const char* fmt, ...);
gs_status from_hip(hipError_t e, const char* what);
bool dtype_ok(gs_dtype d);
int dtype_bytes(gs_dtype d);
int val_bytes_of(gs_dtype d);
// Resolves the no-allocation entry's fixed workspace on `device` (current).
hipError_t noalloc_setup(int device);
gs_status sort_device(gs_handle* h, gs_dtype kdt, void* d_keys, gs_dtype vdt, void* d_vals, uint64_t n,
                      int descending);
// dst[i] = src[idx[i]] queued on h->stream, through source regions where that
// pays and its scratch can be had.
hipError_t gather_device(gs_handle* h, int elem_bytes, const void* src, const uint64_t* idx, void* dst, uint64_t n);
// Segmented sort from host offsets, queued on h->stream without waiting;
// `meta` must outlive the queued work; segments of 2^30+ keys are returned
// in `huge` for the caller to sort.
gs_status sort_segments_async(gs_handle* h, gs_dtype kdt, void* d_keys, gs_dtype vdt, void* d_vals,
                              const uint64_t* off, uint32_t nseg, int descending, std::vector<unsigned char>* meta,
                              std::vector<uint32_t>* huge, const SegConfig* config = nullptr);

}  // namespace gs

struct gs_handle {
  int device = 0;
  hipStream_t stream = nullptr;
  // Tile hand-out of the handle's onesweep passes (gs::TilePolicy); the
  // server grants grouped hand-out to one slot at a time.
  int tile_policy = gs::kTilesByStream;
  // Device bytes one host-memory sort may stage (gs_set_host_sort_budget);
  // 0: the device's free memory at the call.
  uint64_t host_budget = 0;
  gs::Arena arena;
  gs::Profiler profiler;
  gs::LaunchTimer* timer() { return profiler.active ? &profiler : nullptr; }
  void* pinned = nullptr;
  size_t pinned_bytes = 0;
  gs::PinnedStage stage;
  std::vector<uint64_t> seg_offsets;  // gs_sort_segments' host copy
  // Size-class configuration of the batched sort per (key, payload) width,
  // set by the autotuner; defaults otherwise.
  std::map<int, gs::SegConfig> seg_tuned;
  gs::SegConfig seg_config(int kb, int vb) const {
    auto it = seg_tuned.find(kb * 16 + vb);
    return it == seg_tuned.end() ? gs::default_seg_config(kb, vb) : it->second;
  }
};

namespace gs {

// Waits for the handle's stream on every way out of a call but the one that has
// waited already (done): what the call queued reads the pinned stage and vectors
// of its frame.  Declared after them.
struct DrainGuard {
  gs_handle* h;
  bool done = false;
  ~DrainGuard() {
    if (!done) (void)hipStreamSynchronize(h->stream);
  }
};

}  // namespace gs
