// Where the small transfers of a call lie in the handle's pinned buffer, and
// reads of several blocks through it.  No HIP in here: the same code runs
// against plain memory in a CPU test.
#pragma once

#include <stddef.h>
#include <string.h>

#include <initializer_list>
#include <vector>

namespace gs {

// Places in a buffer, handed out front to back.  Past its end the hand-out
// starts over, and every place given before is free for reuse: whatever was
// queued on them must be done (drain), and what a read left there taken out.
// Blocks that are in use together therefore share one place.
class StageRing {
 public:
  static constexpr size_t kNone = ~(size_t)0;
  explicit StageRing(size_t capacity) : capacity_(capacity) {}
  static size_t aligned(size_t bytes) { return ((bytes ? bytes : 1) + 255) & ~(size_t)255; }
  // Offset of a place of `bytes`; kNone if it is larger than the buffer or
  // drain() fails.
  template <typename Drain>
  size_t take(size_t bytes, Drain drain) {
    if (bytes > capacity_ || aligned(bytes) > capacity_) return kNone;
    bytes = aligned(bytes);
    if (used_ + bytes > capacity_) {
      if (!drain()) return kNone;
      used_ = 0;
    }
    used_ += bytes;
    return used_ - bytes;
  }
  void restart() { used_ = 0; }

 private:
  size_t capacity_, used_ = 0;
};

struct ReadBlock {
  void* dst;
  const void* src;
  size_t bytes;
};

// Reads blocks of device memory to host memory: all of them through one place
// of take(bytes), or each straight to its destination if there is none.
// copy(dst, src, bytes) queues a copy, wait() waits for all that is queued;
// both return an error code whose zero is success.
template <typename Take, typename Copy, typename Wait>
auto read_staged(std::initializer_list<ReadBlock> blocks, Take take, Copy copy, Wait wait) -> decltype(wait()) {
  size_t total = 0;
  for (const ReadBlock& b : blocks)
    if (b.bytes) total += StageRing::aligned(b.bytes);
  char* const place = total ? static_cast<char*>(take(total)) : nullptr;
  size_t at = 0;
  for (const ReadBlock& b : blocks) {
    if (b.bytes == 0) continue;
    const auto e = copy(place ? place + at : b.dst, b.src, b.bytes);
    if (e != decltype(e)(0)) return e;
    at += StageRing::aligned(b.bytes);
  }
  const auto e = wait();
  if (e != decltype(e)(0) || !place) return e;
  at = 0;
  for (const ReadBlock& b : blocks) {
    if (b.bytes == 0) continue;
    memcpy(b.dst, place + at, b.bytes);
    at += StageRing::aligned(b.bytes);
  }
  return e;
}

}  // namespace gs
