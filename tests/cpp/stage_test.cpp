// Reads of one to three blocks through a pinned stage, on plain memory: copies
// are queued and done only when the stage drains or the reader waits, as a
// device does them, so a place given out twice shows as a wrong block.
//   stage_test <capacity> <rounds> <seed>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <random>
#include <vector>

#include "../../gpusort_amd/csrc/pinned_stage.h"

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const size_t cap = strtoull(argv[1], nullptr, 10);
  const int rounds = atoi(argv[2]);
  std::mt19937_64 rng(strtoull(argv[3], nullptr, 10));
  std::vector<char> buf(cap);
  gs::StageRing ring(cap);
  struct Copy {
    void* dst;
    const void* src;
    size_t bytes;
  };
  std::vector<Copy> queue;
  auto run_queue = [&] {
    for (const Copy& c : queue) memcpy(c.dst, c.src, c.bytes);
    queue.clear();
    return 0;
  };
  int staged = 0, direct = 0, drains = 0;
  auto take = [&](size_t bytes) -> void* {
    const size_t at = ring.take(bytes, [&] {
      ++drains;
      run_queue();
      return true;
    });
    if (at == gs::StageRing::kNone) {
      ++direct;
      return nullptr;
    }
    if (at % 256 || at + bytes > cap) {
      printf("place %zu + %zu past the buffer\n", at, bytes);
      exit(1);
    }
    ++staged;
    return buf.data() + at;
  };
  auto copy = [&](void* d, const void* s, size_t n) {
    queue.push_back({d, s, n});
    return 0;
  };
  for (int r = 0; r < rounds; ++r) {
    // An upload in between moves the hand-out on, as a plan's does.
    if (rng() % 2) take(rng() % (cap / 3) + 1);
    std::vector<std::vector<char>> src(3), dst(3);
    for (int i = 0; i < 3; ++i) {
      // Empty, a few bytes, half the buffer, or up to more than all of it.
      const size_t kinds[] = {0, (size_t)(rng() % 700), cap / 2 - 256 + (size_t)(rng() % 512), (size_t)(rng() % (cap + cap / 8))};
      src[i].resize(kinds[rng() % 4]);
      for (char& c : src[i]) c = (char)rng();
      dst[i].assign(src[i].size(), 0);
    }
    const int e = gs::read_staged({{dst[0].data(), src[0].data(), src[0].size()},
                                   {dst[1].data(), src[1].data(), src[1].size()},
                                   {dst[2].data(), src[2].data(), src[2].size()}},
                                  take, copy, run_queue);
    if (e != 0 || dst != src) {
      printf("round %d: blocks of %zu, %zu, %zu bytes came back wrong\n", r, src[0].size(), src[1].size(), src[2].size());
      return 1;
    }
  }
  printf("staged %d direct %d drains %d\n", staged, direct, drains);
  return staged && direct && drains ? 0 : 1;
}
