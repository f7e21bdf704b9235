// Radix sorts of 64-bit keys by their highest digits, and the two kernels
// that finish them.
//
// n random 64-bit keys are told apart by little more than log2(n) bits: after
// LSD passes over the highest 32 bits of 2^21 of them, about 500 pairs are
// still equal in the sorted bits.  So the passes start at digit `low` (chosen
// from a sorted sample of the keys, choose_low) and leave short runs of keys
// that agree from bit 8 * low up, in input order.  tie_fix_kernel reads the
// keys once and puts runs of up to kShortRun keys in order by comparing them; runs
// longer than that with a key out of order (keys that share their high digits:
// small numbers or a hot prefix among random ones) are listed and sorted by
// long_run_kernel, in LDS where they fit and by all workgroups together where
// not.  Every step is stable, no step depends on the sample being right, and
// nothing is read back by the host.
//
// What bounds them: tie_fix_kernel the read of the keys (0.23 ms for 2^27
// keys, 4.7 TB/s).  Measured: 2^27 u64 keys + u32 payloads in 64 segments, 8
// passes and their histogram 5.46 ms, 4 passes, theirs and both kernels 3.1 ms;
// one array of 2^26 such pairs 2.94 -> 1.69 ms, of 10^6 0.198 -> 0.114; 2^25
// normal f64 keys + i64 payloads (six digits) 2.03 -> 1.62 ms; Zipf(1.1) u64
// keys 2^24 0.735 -> 0.472.  Where no digit can be left out the sample and the
// idle launches cost about 5 us.  2^26 u64 keys + u32 payloads that share their
// upper half, against 2.9 ms by all digits: one key in twenty 2.2 ms; half of
// them equal but for a few small numbers, which no sample met, 2.5; but for a few
// whose whole lower half differs 3.6, the worst there is (2^18: 0.22, by all
// digits 0.14).
#pragma once

#include <algorithm>
#include <cstddef>

#include "block_radix.h"
#include "gs_device.h"
#include "gs_internal.h"

namespace gs {

// Keys of the sample that picks the lowest digit, and the least n for twice, four and
// eight times as many: a sample of S keys shows clusters of r keys that share their
// high digits by about S^2 r / 2n pairs, and from r = 64 on all digits cost less.
constexpr uint32_t kLowSample = 1024;
constexpr uint64_t kLowSample2Min = 1ull << 24, kLowSample4Min = 1ull << 26, kLowSample8Min = 1ull << 28;
// Digits are added until the sample's ties come to at most 1 in kTieFrac.
// (Gaps of random keys vary, and 1 / gap is counted: 1 in 8 here is about 1
// key in 32 that agrees with another one in the sorted bits.)
constexpr uint32_t kTieFrac = 8;
constexpr uint32_t kShortRun = 256;

// The sample in a workgroup.
template <uint32_t S>
struct LowTileOf {
  static constexpr int THREADS = S < 4096 ? S / 4 : 1024, ITEMS = S / THREADS;
  using T = BlockRadix<uint64_t, uint32_t, false, THREADS, ITEMS, false>;
};

// Position of sample i of S of n keys: one in each of S equal strata, at a place
// of its own.
template <uint32_t S>
__device__ inline uint64_t sample_pos(uint32_t i, uint64_t n) {
  const uint64_t lo = (uint64_t)i * n / S, hi = (uint64_t)(i + 1) * n / S;
  uint32_t x = i * 0x9E3779B1u;
  x ^= x >> 15;
  x *= 0x85EBCA77u;
  x ^= x >> 13;
  return lo + (((hi - lo) * (uint64_t)(x >> 16)) >> 16);
}

// Arrays below this many keys leave out no digit that would put more than a few
// thousand keys into long runs: the runs that workgroups share cost a dozen
// phases of 7-10 us whatever their length (2^22 pairs, 5 % of which share their
// upper half: 0.37 ms, by all digits 0.33; 2^24 0.88 and 0.92).
constexpr uint64_t kSharedMin = 1ull << 23;
constexpr uint32_t kLdsRun = 4096;

// Lowest digit to sort by, from a sample of S of the n keys at `keys`: the largest
// low for which few keys are expected to agree with another one from bit 8 * low
// up, among those that leave out a digit that varies and leave an even number of
// varying ones (the result then lands where the keys were); 0 if none.
// `even_only`: every digit from low up is a pass, so low itself is even.
//
// The n / S keys between two neighbouring samples are taken as spread evenly over
// the gap between them; equal samples are taken as equal keys.  Samples that agree
// from bit 8 * low up but differ below stand for one run, all of them: half of 2^26
// keys in 0..99, which as 99 gaps among 1024 looked like few, went to one
// workgroup (480 ms, by all digits 2.9).  Two of them with no third stand for many
// small clusters, of about 2 n / S^2 keys for every such pair: more than kMaxMates
// keys are more than is worth comparing (2^26 keys in 2^20 clusters: 51 ms).
//
// All threads of the workgroup; every one returns the answer.  About 9 us alone on
// the chip with 1024 samples, of which their reads are 2; 15, 26 and 42 with 2048,
// 4096 and 8192.
constexpr uint32_t kMaxMates = 64;

template <uint32_t S>
__device__ inline uint32_t choose_low(typename LowTileOf<S>::T::Smem& sm, const uint64_t* __restrict__ keys, uint64_t n,
                                      const Xform<uint64_t>& xf, bool even_only, uint32_t* s_sum) {
  using LowTile = typename LowTileOf<S>::T;
  constexpr int THREADS = LowTileOf<S>::THREADS, ITEMS = LowTileOf<S>::ITEMS;
  const uint32_t tid = threadIdx.x;
  uint64_t k[ITEMS];
  uint32_t none[1];
  LowTile t{sm, k, none, S, (uint32_t)ITEMS};
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) k[i] = to_ordered(keys[sample_pos<S>(t.pos(i), n)], xf);
  if (tid < 24) s_sum[tid] = 0;
  const uint64_t diff = t.varying();
  uint32_t allowed = 0, above = 0;
  for (int p = 7; p > 0; --p) {
    above += ((diff >> (8 * p)) & 0xFFu) ? 1u : 0u;
    if (above >= 2 && !((even_only ? (uint32_t)p : above) & 1u) && (diff & ((1ull << (8 * p)) - 1))) allowed |= 1u << p;
  }
  if (allowed == 0) return 0;
  lds_barrier();  // every thread has read what varying() left
  t.sort();
  lds_barrier();
  const uint64_t* const sk = t.keys();
  const float per = (float)n * (4096.0f / (float)S);
  // This thread's gaps: the ties expected at low = 0, in 1/4096 of a sample (256
  // times as many with every digit, up to the whole sample), and the lowest low at
  // which the samples on both sides agree.
  float ties[ITEMS];
  uint32_t next[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t p = tid + (uint32_t)j * THREADS;
    ties[j] = 0.0f;
    next[j] = 8;
    if (p + 1 < S) {
      // The staged samples are in order but for a few neighbours: those count
      // as close ones.
      const uint64_t a = sk[p], b = sk[p + 1];
      if (a != b) {
        ties[j] = per * __builtin_amdgcn_rcpf(b > a ? (float)(b - a) : 1.0f);
        next[j] = 8 - (uint32_t)__clzll((long long)(a ^ b)) / 8;
      }
    }
  }
#pragma unroll
  for (uint32_t low = 1; low < 8; ++low) {
    if (!((allowed >> low) & 1u)) continue;
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) sum += fminf(ties[j] * (float)(1ull << (8 * low)), 4096.0f);
    const uint32_t w = wave_incl_scan_dpp((uint32_t)sum);
    if ((tid & 63u) == 63u) atomicAdd(&s_sum[low], w);
  }
  lds_barrier();
  constexpr uint32_t kMost = 4096u * S / kTieFrac;
  uint32_t prev[ITEMS], size[ITEMS];
  bool sized = false;
  for (uint32_t low = 7; low > 0; --low) {
    if (!((allowed >> low) & 1u) || s_sum[low] > kMost) continue;
    uint32_t pairs = 0;  // different samples side by side in one run
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) pairs += next[j] <= low ? 1u : 0u;
    if (!__syncthreads_or((int)pairs)) return low;
    if (!sized) {
      // Equal samples that end at this thread's places: how many, and the lowest
      // low at which they agree with the different ones before them.
      sized = true;
      uint64_t* const ends = reinterpret_cast<uint64_t*>(t.counts());  // a bit for every sample whose next one differs
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        const uint64_t w = ballot(ties[j] != 0.0f);
        if ((tid & 63u) == 0) ends[(tid + (uint32_t)j * THREADS) / 64] = w;
      }
      lds_barrier();
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        const uint32_t p = tid + (uint32_t)j * THREADS;
        prev[j] = 8;
        size[j] = 0;
        if (ties[j] == 0.0f && p + 1 < S) continue;
        int w = (int)(p / 64);
        uint64_t before = ends[w] & ((1ull << (p % 64)) - 1);
        while (before == 0 && w > 0) before = ends[--w];
        const int last = before ? w * 64 + 63 - __clzll((long long)before) : -1;
        size[j] = (uint32_t)((int)p - last);
        if (last >= 0) prev[j] = 8 - (uint32_t)__clzll((long long)(sk[last] ^ sk[last + 1])) / 8;
      }
    }
    uint32_t mixed = 0, alone = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      mixed += next[j] <= low || prev[j] <= low ? size[j] : 0u;
      if (next[j] <= low) {  // the pair p, p + 1: has it a third?
        const uint32_t p = tid + (uint32_t)j * THREADS;
        const uint64_t g = sk[p] >> (8 * low);
        alone += (p == 0 || (sk[p - 1] >> (8 * low)) != g) && (p + 2 >= S || (sk[p + 2] >> (8 * low)) != g) ? 1u : 0u;
      }
    }
    const uint32_t m = wave_incl_scan_dpp(mixed), c = wave_incl_scan_dpp(pairs), l = wave_incl_scan_dpp(alone);
    if ((tid & 63u) == 63u) {
      atomicAdd(&s_sum[8 + low], m - 2 * l);
      atomicAdd(&s_sum[16 + low], l);
      atomicAdd(&s_sum[low], 4096u * (m - c));  // such a pair counted as one
    }
    lds_barrier();
    const uint64_t clusters = s_sum[16 + low];
    if (s_sum[low] <= kMost && (n >= kSharedMin || s_sum[8 + low] * n <= (uint64_t)kLdsRun * S) &&
        (clusters <= 2 || clusters * n <= (uint64_t)S * S * (kMaxMates / 2)))
      return low;
  }
  return 0;
}

// Keys a thread of long_run_kernel's LDS tile: what fits the registers without
// spills.  Longer runs are cut into chunks that workgroups share.
template <typename V, bool KV>
constexpr uint32_t run_items() {
  return !KV ? 12 : sizeof(V) == 4 ? 8 : 6;
}
constexpr uint32_t kRunChunk = 4096;

struct SharedRun {
  uint64_t start, len;
  unsigned long long diff;  // bits that vary in it
  uint32_t chunk0;          // its first chunk among those of all shared runs
  uint32_t pad;
};
static_assert(sizeof(SharedRun) == 32, "the size that use_status reckons with");

// Words of the control block that they start from zero.
constexpr uint32_t kTieWords = (sizeof(SortCtrl) - offsetof(SortCtrl, top_digits)) / 4;

// Where the keys are: one array of n keys (tile_seg null) or the segments of a
// segmented sort, in buffer 0.
template <typename V>
struct TieArgs {
  uint64_t* keys0;
  uint64_t* keys1;
  V* vals0;
  V* vals1;
  uint64_t n;
  Xform<uint64_t> xf;
  SortCtrl* ctrl;
  uint32_t tile_keys;
  const uint32_t* tile_seg;
  const uint32_t* seg_first;
  const uint64_t* seg_range;
  // Long runs, each at least kShortRun + 1 keys: a bit for every 32 positions
  // of every tile (zeroed); those that fit an LDS tile, three words each (start
  // and slot); the others; and, from its end down, their chunks' digit counts.
  uint32_t* long_seen;
  uint32_t* long_list;
  SharedRun* shared;
  void* rows_end;

  // They take the look-back words, which are done with by then: the bits and
  // the shared runs those of pass 0 (left out whenever the kernels have work, so
  // still zero), the list and the counts the following passes'.
  template <uint32_t TILE, bool KV, typename S>
  void use_status(S* status, uint64_t tiles) {
    constexpr uint64_t kPass = 256, CAP = 1024 * run_items<V, KV>();
    // Per tile: bits, and runs longer than CAP.
    static_assert(TILE / 256 + 64 + 32 * (TILE / CAP + 1) <= kPass * sizeof(uint32_t), "bits and shared runs fit a pass");
    // All keys in the shortest listed runs, or all in the shortest shared ones;
    // what lies between is a mixture of the two.
    static_assert((TILE / (kShortRun + 1) + 1) * 12 <= 7 * kPass * sizeof(uint32_t), "listed runs fit seven passes");
    static_assert(TILE / (kRunChunk / 256) * sizeof(uint32_t) + kPass * sizeof(uint32_t) * TILE / CAP <=
                      7 * kPass * sizeof(uint32_t),
                  "the chunks' counts fit seven passes");
    long_seen = reinterpret_cast<uint32_t*>(status);
    shared = reinterpret_cast<SharedRun*>(reinterpret_cast<char*>(status) + align_up((tiles * TILE / 1024 + 1) * 4, 64));
    long_list = reinterpret_cast<uint32_t*>(status + tiles * kPass);
    rows_end = status + 8 * tiles * kPass;
  }
};

// First position in [lo, hi) whose key agrees with t from bit s up or is
// greater (the keys are in order from bit s up).
__device__ inline uint64_t first_at_least(const uint64_t* keys, uint64_t lo, uint64_t hi, uint64_t t, int s,
                                          const Xform<uint64_t>& xf) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if ((to_ordered(keys[mid], xf) >> s) < t)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Puts runs of 2..kShortRun keys equal from bit 8 * ctrl->low() up in order,
// and lists longer runs that hold a key out of order.  A workgroup takes
// chunks of kTieChunk keys, staged in LDS with the kShortRun keys behind them (all
// loads in flight together).  A bit is set for every key that starts a run and for
// every key greater than the next one of its run; where none of the latter is near,
// nothing is done, so equal keys cost nothing.  The keys in runs near one are
// collected, so that the work is by such keys, and each finds the ends of its run
// from the bits and its place by comparison with all keys of the run.  Payloads are
// read before any is written.  A run belongs to the chunk it starts in.  Where a run
// starts and ends depends only on bits that no step changes, so a run has one owner
// and reads of other owners' keys decide nothing about it.
//
// What bounds it: the read of the keys (2^26 random keys, 1.5 % of them in runs, with
// 32-bit payloads: 200 us); where all keys are in runs of r keys, the r LDS reads
// a key (r = 4: 0.7 ms, 16: 0.8, 32: 1.0, 64: 1.3).  With a thread a run up to 32
// keys, in global memory, and a workgroup a run above, the sort of those 2^26 took
// 13.3 ms at r = 16 and 51 at 64 (now 2.4 and 3.0; by all digits 2.9).  120 registers,
// four workgroups a CU; five, with two registers spilled, or the next chunk's loads
// ahead, are slower (keys only: 152 us, 157, 183).
constexpr uint32_t kTieChunk = 2048;

template <typename V, bool KV>
__global__ __launch_bounds__(256) void tie_fix_kernel(TieArgs<V> a) {
  constexpr int PER = (kTieChunk + kShortRun) / 256;
  constexpr uint32_t PAD = kShortRun / 64, WORDS = (kTieChunk + kShortRun) / 64;
  static_assert(kShortRun % 256 == 0 && WORDS < 64, "whole rounds of the workgroup, a word a lane");
  __shared__ uint64_t s_k[kTieChunk + kShortRun + 1];  // from one key before the chunk
  __shared__ uint64_t s_down[WORDS], s_start[WORDS];
  __shared__ alignas(16) uint32_t s_any[4];
  __shared__ uint32_t s_list[kTieChunk + kShortRun];  // place, and the new one in the upper half
  const uint32_t low = a.ctrl->low();
  if (low == 0) return;
  const int s = 8 * (int)low;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  uint64_t seg0 = 0, seg1 = a.n, start, end;
  uint32_t slot = 0;
  uint64_t* keys = a.keys0;
  V* vals = a.vals0;
  if (a.tile_seg) {
    slot = a.tile_seg[blockIdx.x];
    seg0 = a.seg_range[2 * slot];
    seg1 = a.seg_range[2 * slot + 1];
    start = seg0 + (uint64_t)(blockIdx.x - a.seg_first[slot]) * a.tile_keys;
  } else {
    start = (uint64_t)blockIdx.x * a.tile_keys;
  }
  end = start + a.tile_keys < seg1 ? start + a.tile_keys : seg1;
  // Element i of the chunk.
  auto at = [&](uint32_t i) -> uint64_t& { return s_k[i + 1]; };
  for (uint64_t c0 = start; c0 < end; c0 += kTieChunk) {
    const uint32_t m = end - c0 < kTieChunk ? (uint32_t)(end - c0) : kTieChunk;
    const uint32_t staged = seg1 - c0 < m + kShortRun ? (uint32_t)(seg1 - c0) : m + kShortRun;
    uint64_t k[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      k[j] = keys[c0 + (i < staged ? i : staged - 1)];
    }
    // Before the segment: a key of another run.
    if (tid == 64) s_k[0] = c0 > seg0 ? to_ordered(keys[c0 - 1], a.xf) : ~to_ordered(keys[c0], a.xf);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      k[j] = to_ordered(k[j], a.xf);
      if (i < staged) at(i) = k[j];
    }
    lds_barrier();
    uint64_t down[PER], any = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      const uint64_t next = at(i + 1 < staged ? i + 1 : staged - 1);
      down[j] = ballot(next < k[j] && ((next ^ k[j]) >> s) == 0);
      any |= down[j];
    }
    if (lane == 0) s_any[tid / 64] = any != 0;
    lds_barrier();
    const uint4 found = *reinterpret_cast<const uint4*>(s_any);
    if (__builtin_amdgcn_readfirstlane((int)(found.x | found.y | found.z | found.w)) == 0) continue;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      const uint64_t starts = ballot(i >= staged || ((s_k[i] ^ k[j]) >> s) != 0);
      if (lane == 0) {
        s_down[i / 64] = down[j];
        s_start[i / 64] = starts;
      }
    }
    lds_barrier();
    // A lane a word: the keys of it that are in a run, if a bit is within kShortRun.
    const uint64_t downs = ballot(lane < WORDS && s_down[lane < WORDS ? lane : 0] != 0);
    uint64_t in_run = 0;
    if (lane < WORDS && ((lane >= PAD ? downs >> (lane - PAD) : downs << (PAD - lane)) & ((1u << (2 * PAD + 1)) - 1))) {
      const uint64_t st = s_start[lane], next = lane + 1 < WORDS ? s_start[lane + 1] : ~0ull;
      in_run = ~st | ~((st >> 1) | (next << 63));
    }
    const uint32_t incl = wave_incl_scan_dpp((uint32_t)__popcll(in_run));
    const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      const int w = __builtin_amdgcn_readfirstlane((int)(i / 64));
      const uint64_t bits = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)in_run, w) |
                            (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(in_run >> 32), w) << 32;
      const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)incl, w) - (uint32_t)__popcll(bits);
      if ((bits >> lane) & 1u) s_list[before + (uint32_t)__popcll(bits & ((1ull << lane) - 1))] = i;
    }
    lds_barrier();
    for (uint32_t q = tid; q < count; q += 256) {
      const uint32_t i = s_list[q];
      const uint64_t x = at(i), t = x >> s;
      s_list[q] = i | i << 16;
      // The run [b, e) as far as it is within kShortRun keys.
      int w = (int)(i / 64);
      uint64_t bits = s_start[w] & (~0ull >> (63 - i % 64));
      for (const int last = w > (int)PAD ? w - (int)PAD : 0; bits == 0 && w > last;) bits = s_start[--w];
      const bool starts = bits != 0;
      const uint32_t b = starts ? (uint32_t)(w * 64 + 63 - __clzll((long long)bits)) : 0;
      w = (int)(i / 64);
      bits = s_start[w] & ~(~0ull >> (63 - i % 64));
      for (const int last = w + (int)PAD < (int)WORDS - 1 ? w + (int)PAD : (int)WORDS - 1; bits == 0 && w < last;)
        bits = s_start[++w];
      uint32_t e = bits ? (uint32_t)(w * 64) + (uint32_t)__ffsll((unsigned long long)bits) - 1u : staged;
      if (e > staged) e = staged;
      // Whether a key of [from, to) is greater than the next of the run.
      auto unordered = [&](uint32_t from, uint32_t to) {
        uint64_t found = 0;
        for (uint32_t v = from / 64; v <= to / 64 && v < WORDS; ++v) {
          uint64_t d = s_down[v];
          if (v == from / 64) d &= ~0ull << (from % 64);
          if (v == to / 64) d &= (1ull << (to % 64)) - 1;
          found |= d;
        }
        return found != 0;
      };
      if (starts && e - b <= kShortRun) {
        if (b >= m || !unordered(b, e)) continue;  // the next chunk's
        uint32_t rank = b;
#pragma unroll 4
        for (uint32_t p = b; p < e; ++p) {
          const uint64_t y = at(p);
          rank += y < x || (y == x && p < i) ? 1u : 0u;
        }
        s_list[q] = i | rank << 16;
        continue;
      }
      // A long run, or one that starts before the chunk.  An earlier key of it that
      // is greater than the next asks in its place.
      if (i >= m || !((s_down[i / 64] >> (i % 64)) & 1u)) continue;
      const uint32_t seen = starts ? b : i > kShortRun ? (i / 64 - PAD) * 64 : 0;
      if (unordered(seen, i)) continue;
      uint64_t run = c0 + b;
      if (!starts) {
        const uint64_t p = c0 + i;
        const uint64_t back = p - seg0 > kShortRun ? p - kShortRun : seg0;
        const uint64_t fwd = seg1 - p > kShortRun + 1 ? p + kShortRun + 1 : seg1;
        const uint64_t rb = first_at_least(keys, back, p, t, s, a.xf);
        const uint64_t re = first_at_least(keys, p + 1, fwd, t + 1, s, a.xf);
        if (re - rb <= kShortRun) continue;
        run = rb > back ? rb : first_at_least(keys, seg0, rb, t, s, a.xf);
      }
      // Two runs longer than kShortRun never start in the same 32 positions.
      const uint64_t place = a.tile_seg ? (uint64_t)a.seg_first[slot] * a.tile_keys + (run - seg0) : run;
      const uint32_t bit = 1u << ((place >> 5) & 31u);
      if (atomicOr(&a.long_seen[place >> 10], bit) & bit) continue;
      constexpr uint64_t CAP = 1024 * run_items<V, KV>();
      if (seg1 - run > CAP && (to_ordered(keys[run + CAP], a.xf) >> s) == t) {
        const uint64_t len = first_at_least(keys, run + CAP + 1, seg1, t + 1, s, a.xf) - run;
        const uint64_t chunks = (len + kRunChunk - 1) / kRunChunk;
        const unsigned long long was = atomicAdd(&a.ctrl->shared, (1ull << 32) + chunks);
        a.shared[was >> 32] = SharedRun{run, len, 0, (uint32_t)was, 0};
        continue;
      }
      uint32_t* const entry = a.long_list + 3 * (uint64_t)atomicAdd(&a.ctrl->long_count, 1u);
      entry[0] = (uint32_t)run;
      entry[1] = (uint32_t)(run >> 32);
      entry[2] = slot;
    }
    // This thread's keys of the list.
    uint32_t move[PER];
    V v[KV ? PER : 1];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t q = tid + (uint32_t)j * 256;
      move[j] = q < count ? s_list[q] : 0;
      if constexpr (KV)
        if (move[j] >> 16 != (move[j] & 0xFFFFu)) v[j] = vals[c0 + (move[j] & 0xFFFFu)];
    }
    __syncthreads();  // every payload that moves is read
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = move[j] & 0xFFFFu, dst = move[j] >> 16;
      if (dst == i) continue;
      keys[c0 + dst] = from_ordered(at(i), a.xf);
      if constexpr (KV) vals[c0 + dst] = v[j];
    }
    lds_barrier();  // the chunk's keys are read
  }
}

// Sorts the listed runs, a workgroup a run in LDS, and then the shared ones,
// which do not fit a tile, by their digits below ctrl->low() that vary: for each
// digit the chunks' counts, their scan a run, and every chunk sorted by the digit
// in LDS and written behind the chunks before it in the other buffer.
//
// The workgroups take the shared runs' tasks by one ticket, phase after phase,
// and a task waits until the phase before its own is done.  Every task of that
// phase has a lower ticket, so a running workgroup holds it: the kernel finishes
// whatever share of the chip it gets, with no need that all of its workgroups
// run at once.  What the phases pass on crosses XCDs, so a task's writes are
// released, and the ones it reads acquired, at agent scope.
//
// What bounds it: up to a chunk a CU a phase's chain of waits, cache write-backs
// and LDS steps (7-10 us), beyond that the LDS work of the moves (2^25 keys and
// u32 payloads about 0.45 ms a digit).
enum RunTask : uint32_t { kTaskVary, kTaskCount, kTaskScan, kTaskMove, kTaskCopy };

template <typename V, bool KV, typename S>
__global__ __launch_bounds__(1024) void long_run_kernel(TieArgs<V> a) {
  constexpr int ITEMS = run_items<V, KV>();
  using Tile = BlockRadix<uint64_t, V, KV, 1024, ITEMS, true>;
  using Part = BlockRadix<uint64_t, V, KV, 1024, kRunChunk / 1024, false>;
  struct S4 {
    S x, y, z, w;
  };
  __shared__ union {
    typename Tile::Smem tile;
    typename Part::Smem part;
    uint32_t count[256];
    S4 sums[16][64];
    uint64_t diff[16];
  } sm;
  __shared__ S s_off[256];
  __shared__ uint64_t s_end;
  __shared__ uint32_t s_task;
  SortCtrl* const ctrl = a.ctrl;
  const uint32_t count = ctrl->long_count, low = ctrl->low();
  const uint32_t runs = (uint32_t)(ctrl->shared >> 32), chunks = (uint32_t)ctrl->shared;
  if (count == 0 && chunks == 0) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const int s = 8 * (int)low;
  uint64_t* const keys = a.keys0;
  V* const vals = a.vals0;
  for (uint32_t job = blockIdx.x; job < count; job += gridDim.x) {
    const uint32_t* const entry = a.long_list + 3 * (uint64_t)job;
    const uint64_t p0 = entry[0] | (uint64_t)entry[1] << 32;
    if (tid == 0) {
      const uint64_t seg1 = a.tile_seg ? a.seg_range[2 * entry[2] + 1] : a.n;
      const uint64_t stop = seg1 - p0 > Tile::CAP ? p0 + Tile::CAP : seg1;
      s_end = first_at_least(keys, p0, stop, (to_ordered(keys[p0], a.xf) >> s) + 1, s, a.xf);
    }
    __syncthreads();
    const uint32_t m = (uint32_t)(s_end - p0);
    uint64_t k[ITEMS];
    V v[KV ? ITEMS : 1];
    Tile t{sm.tile, k, v, m, (m + 1023) / 1024};
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t p = t.pos(i);
      const bool in = (uint32_t)i < t.items && p < m;
      k[i] = in ? to_ordered(keys[p0 + p], a.xf) : ~0ull;
      if constexpr (KV) v[i] = in ? vals[p0 + p] : V(0);
    }
    const int at = t.sort();
    if (at != Tile::kInOrder) {
      const V* const sv = t.vals();
      t.write_out(at, [&](uint32_t dst, uint64_t x, uint32_t p) {
        keys[p0 + dst] = from_ordered(x, a.xf);
        if constexpr (KV) vals[p0 + dst] = sv[p];
      });
    }
    __syncthreads();
  }

  if (chunks == 0) return;
  S* const rows = reinterpret_cast<S*>(a.rows_end) - (uint64_t)chunks * 256;
  // A task takes `group` chunks, so that a phase is about one task a workgroup.
  const uint32_t group = (chunks + gridDim.x - 1) / gridDim.x, tasks = (chunks + group - 1) / group;
  // Everything that decides a branch around a barrier is read into scalar
  // registers: a loop of tasks that lanes leave and enter one by one is one that
  // part of a wave may go round in, through the barrier, without the others.
  const uint32_t wave0 = __builtin_amdgcn_readfirstlane(wave);
  auto load_now = [](const uint32_t* p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane(
        __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  auto diff_of = [](const unsigned long long* p) {
    const uint64_t x = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32)) << 32 |
           (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
  };
  // Waits until `n` tasks of a phase are done; what they wrote is visible then:
  // one wave invalidates the caches that the workgroup reads through, and is
  // done with it before the others go on (an acquire in each of the 16 waves is
  // 10 us a phase more).
  auto wait = [&](uint32_t phase, uint32_t n) {
    if (wave0 == 0) {
      while (load_now(&ctrl->done[phase]) < n) __builtin_amdgcn_s_sleep(4);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
  };
  // Digits below `digit` in which bits of `diff` are set.
  auto digits_in = [](uint64_t diff, uint32_t digit) {
    uint32_t c = 0;
    for (uint32_t d = 0; d < digit; ++d) c += (diff >> (8 * d)) & 0xFFu ? 1u : 0u;
    return c;
  };
  // Counts -> offsets in the run, digit by digit and task by task: a wave a
  // sixteenth of the rows, four digits a lane.
  auto scan_run = [&](const SharedRun& run, uint32_t digit) {
    if (((diff_of(&run.diff) >> (8 * digit)) & 0xFFu) == 0) return;
    const uint32_t chunk0 = run.chunk0, last = chunk0 + (uint32_t)((run.len - 1) / kRunChunk);
    const uint32_t task0 = chunk0 / group, n = last / group - task0 + 1;
    // Row of the i-th task of the run: that of the task's first chunk in it.
    auto row = [&](uint32_t i) -> S4& {
      const uint32_t c = i ? (task0 + i) * group : chunk0;
      return reinterpret_cast<S4*>(rows + (uint64_t)c * 256)[lane];
    };
    constexpr int UN = sizeof(S) == 4 ? 8 : 4;
    const uint32_t r0 = (uint32_t)((uint64_t)n * wave / 16), r1 = (uint32_t)((uint64_t)n * (wave + 1) / 16);
    S4 sum{0, 0, 0, 0};
#pragma unroll UN
    for (uint32_t i = r0; i < r1; ++i) {
      const S4 c = row(i);
      sum.x += c.x;
      sum.y += c.y;
      sum.z += c.z;
      sum.w += c.w;
    }
    sm.sums[wave][lane] = sum;
    __syncthreads();
    if (wave == 0) {
      S4 all{0, 0, 0, 0};
#pragma unroll 2
      for (int w = 0; w < 16; ++w) {
        const S4 c = sm.sums[w][lane];
        all.x += c.x;
        all.y += c.y;
        all.z += c.z;
        all.w += c.w;
      }
      const uint64_t mine = (uint64_t)all.x + all.y + all.z + all.w;
      S4 to;
      to.x = (S)(wave_incl_scan64(mine) - mine);
      to.y = to.x + all.x;
      to.z = to.y + all.y;
      to.w = to.z + all.z;
#pragma unroll 2
      for (int w = 0; w < 16; ++w) {
        const S4 c = sm.sums[w][lane];
        sm.sums[w][lane] = to;
        to.x += c.x;
        to.y += c.y;
        to.z += c.z;
        to.w += c.w;
      }
    }
    __syncthreads();
    S4 to = sm.sums[wave][lane];
    for (uint32_t i = r0; i < r1; i += UN) {
      S4 c[UN];
#pragma unroll
      for (int q = 0; q < UN; ++q)
        if (i + q < r1) c[q] = row(i + q);
#pragma unroll
      for (int q = 0; q < UN; ++q) {
        if (i + q < r1) {
          row(i + q) = to;
          to.x += c[q].x;
          to.y += c[q].y;
          to.z += c[q].z;
          to.w += c[q].w;
        }
      }
    }
  };
  // Chunk `at` of a task that takes chunks [begin, stop), in order.
  auto chunk_task = [&](uint32_t task, uint32_t at, uint32_t begin, uint32_t stop, uint32_t digit) {
    uint32_t r = 0, hi = runs;
    while (hi - r > 1) {
      const uint32_t mid = (r + hi) >> 1;
      if (a.shared[mid].chunk0 <= at)
        r = mid;
      else
        hi = mid;
    }
    SharedRun* const run = &a.shared[r];
    const uint32_t chunk0 = run->chunk0;
    const uint64_t start = run->start, len = run->len, diff = task == kTaskVary ? 0 : diff_of(&run->diff);
    // Every digit that varies in the run has moved it to the other buffer.
    const bool away = digits_in(diff, digit) & 1u;
    const bool varies = ((diff >> (8 * digit)) & 0xFFu) != 0;
    const uint64_t base = start + (uint64_t)(at - chunk0) * kRunChunk, left = start + len - base;
    const uint32_t m = left < kRunChunk ? (uint32_t)left : kRunChunk;
    // The task's chunks of one run share a row, that of the first of them.
    const bool first_of_run = at == begin || at == chunk0, last_of_run = at + 1 == stop || left <= kRunChunk;
    S* const row = rows + (uint64_t)(begin > chunk0 ? begin : chunk0) * 256;
    const uint64_t* const ki = (away ? a.keys1 : a.keys0) + base;
    const V* const vi = (away ? a.vals1 : a.vals0) + base;
    if (task == kTaskVary) {
      const uint64_t x0 = to_ordered(keys[start], a.xf);
      uint64_t d = 0;
#pragma unroll
      for (uint32_t j = 0; j < kRunChunk; j += 1024) d |= to_ordered(ki[j + tid < m ? j + tid : 0], a.xf) ^ x0;
      const uint32_t d0 = wave_or_dpp((uint32_t)d), d1 = wave_or_dpp((uint32_t)(d >> 32));
      if (lane == 63) sm.diff[wave] = (uint64_t)d1 << 32 | d0;
      __syncthreads();
      if (tid == 0) {
        for (int w = 1; w < 16; ++w) d |= sm.diff[w];
        d |= sm.diff[0];
        if (d & ~diff_of(&run->diff)) atomicOr(&run->diff, (unsigned long long)d);
        if (d & ~diff_of(&ctrl->shared_diff)) atomicOr(&ctrl->shared_diff, (unsigned long long)d);
      }
    } else if (task == kTaskCopy) {
      if (away)
        for (uint32_t i = tid; i < m; i += 1024) {
          keys[base + i] = ki[i];
          if constexpr (KV) vals[base + i] = vi[i];
        }
    } else if (!varies) {
      // The digit is the same all over the run: it stays where it is.
    } else if (task == kTaskCount) {
      uint64_t k[kRunChunk / 1024];
#pragma unroll
      for (uint32_t j = 0; j < kRunChunk / 1024; ++j) k[j] = ki[j * 1024 + tid < m ? j * 1024 + tid : 0];
      if (first_of_run && tid < 256) sm.count[tid] = 0;
      lds_barrier();
#pragma unroll
      for (uint32_t j = 0; j < kRunChunk / 1024; ++j)
        if (j * 1024 + tid < m) atomicAdd(&sm.count[digit_of(to_ordered(k[j], a.xf), 8 * (int)digit)], 1u);
      lds_barrier();
      if (last_of_run && tid < 256) row[tid] = sm.count[tid];
    } else {
      if (first_of_run && tid < 256) s_off[tid] = row[tid];
      uint64_t k[kRunChunk / 1024];
      V v[KV ? kRunChunk / 1024 : 1];
      Part t{sm.part, k, v, m, (m + 1023) / 1024};
#pragma unroll
      for (int i = 0; i < (int)kRunChunk / 1024; ++i) {
        const uint32_t p = t.pos(i);
        const bool in = (uint32_t)i < t.items && p < m;
        k[i] = in ? to_ordered(ki[p], a.xf) : ~0ull;
        if constexpr (KV) v[i] = in ? vi[p] : V(0);
      }
      t.clear_masks();
      t.digit(8 * (int)digit);
      // Wave 0's first slots are the digits' starts in the chunk.
      const uint32_t* const first = t.counts();
      const uint64_t* const sk = t.keys();
      const V* const sv = t.vals();
      uint64_t* const ko = (away ? a.keys0 : a.keys1) + start;
      V* const vo = (away ? a.vals0 : a.vals1) + start;
      for (uint32_t p = tid; p < m; p += 1024) {
        const uint64_t x = sk[p];
        const uint32_t dg = digit_of(x, 8 * (int)digit);
        const uint64_t dst = s_off[dg] + (p - first[dg]);
        ko[dst] = from_ordered(x, a.xf);
        if constexpr (KV) vo[dst] = sv[p];
      }
      lds_barrier();
      // Slots past the chunk sit in the last digit.
      if (tid < 256) s_off[tid] += (tid == 255 || first[tid + 1] > m ? m : first[tid + 1]) - (first[tid] < m ? first[tid] : m);
    }
    lds_barrier();  // the LDS is free for the next chunk
  };
  if (tid == 0) s_task = __hip_atomic_fetch_add(&ctrl->task_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  for (;;) {
    // The task in its phase: a group of chunks, or the run of a scan.
    uint32_t at = __builtin_amdgcn_readfirstlane(s_task);
    uint32_t phase = 0, digit = 0, task = kTaskVary;
    if (at >= tasks) {
      wait(0, tasks);
      const uint64_t diff = diff_of(&ctrl->shared_diff);
      const uint32_t varying = digits_in(diff, low), per = 2 * tasks + runs;
      at -= tasks;
      const uint32_t turn = at / per < varying ? at / per : varying;
      at -= turn * per;
      phase = 1 + 3 * turn;
      uint32_t before = tasks;
      if (turn == varying) {
        if (at >= tasks) return;
        task = kTaskCopy;
        digit = low;
      } else {
        while (((diff >> (8 * digit)) & 0xFFu) == 0 || digits_in(diff, digit) < turn) ++digit;
        task = kTaskCount;
        if (at >= tasks + runs) {
          at -= tasks + runs;
          task = kTaskMove;
          phase += 2;
          before = runs;
        } else if (at >= tasks) {
          at -= tasks;
          task = kTaskScan;
          phase += 1;
        }
      }
      wait(phase - 1, before);
    }
    if (task == kTaskScan) {
      scan_run(a.shared[at], digit);
    } else {
      const uint32_t begin = at * group, stop = chunks - begin > group ? begin + group : chunks;
      for (uint32_t c = begin; c < stop; ++c) chunk_task(task, c, begin, stop, digit);
    }
    // Every wave's writes have reached the L2 before one thread writes it back
    // (a release in each of the 16 waves: 88 us a phase).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // and everyone has read s_task
    if (tid == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_fetch_add(&ctrl->done[phase], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_task = __hip_atomic_fetch_add(&ctrl->task_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
  }
}

template <typename V, bool KV, typename S>
void launch_tie_fix(const TieArgs<V>& t, uint64_t tiles, uint64_t n_keys, hipStream_t stream, LaunchTimer* timer,
                    const SortCtrl* watched) {
  if (timer) {
    timer->begin("tie_fix", n_keys * 8, stream);
    timer->only_if(watched, LaunchTimer::kTiePass);
  }
  hipLaunchKernelGGL((tie_fix_kernel<V, KV>), dim3((uint32_t)tiles), dim3(256), 0, stream, t);
  if (timer) {
    timer->end(stream);
    timer->begin("long_run", 0, stream);  // its bytes depend on the keys
    timer->only_if(watched, LaunchTimer::kTiePass);
  }
  hipLaunchKernelGGL((long_run_kernel<V, KV, S>), dim3((uint32_t)std::min<uint64_t>(256, n_keys / 16384 + 1)),
                     dim3(1024), 0, stream, t);
  if (timer) timer->end(stream);
}

}  // namespace gs
