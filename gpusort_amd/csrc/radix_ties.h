// Radix sorts of 64-bit keys by their highest digits, and the two kernels
// that finish them.
//
// n random 64-bit keys are told apart by little more than log2(n) bits: after
// LSD passes over the highest 32 bits of 2^21 of them, about 500 pairs are
// still equal in the sorted bits.  So the passes start at digit `low` (chosen
// from a sorted sample of the keys, choose_low) and leave short runs of keys
// that agree from bit 8 * low up, in input order.  tie_fix_kernel reads the
// keys once and puts runs of up to kShortRun keys in order in place; runs
// longer than that with a key out of order (heavy duplicates that share their
// high digits with another value) are listed and sorted by a workgroup each
// (long_run_kernel).  Every step is stable, no step depends on the sample
// being right, and nothing is read back by the host.
//
// What bounds them: tie_fix_kernel the read of the keys (0.23 ms for 2^27
// keys, 4.7 TB/s).  Measured: 2^27 u64 keys + u32 payloads in 64 segments, 8
// passes and their histogram 5.46 ms, 4 passes, theirs and both kernels 3.1 ms;
// one array of 2^26 such pairs 2.94 -> 1.69 ms, of 10^6 0.198 -> 0.114; 2^25
// normal f64 keys + i64 payloads (six digits) 2.03 -> 1.62 ms; Zipf(1.1) u64
// keys 2^24 0.735 -> 0.472.  Where no digit can be left out the sample and the
// idle launches cost about 5 us.
#pragma once

#include <algorithm>

#include "block_radix.h"
#include "gs_device.h"
#include "gs_internal.h"

namespace gs {

// Keys of the sample that picks the lowest digit.
constexpr uint32_t kLowSample = 1024;
// Digits are added until the sample's ties come to at most 1 in kTieFrac.
// (Gaps of random keys vary, and 1 / gap is counted: 1 in 8 here is about 1
// key in 32 that agrees with another one in the sorted bits.)
constexpr uint32_t kTieFrac = 8;
constexpr uint32_t kShortRun = 32;

using LowTile = BlockRadix<uint64_t, uint32_t, false, 256, 4, false>;

// Position of sample i of n keys: one in each of kLowSample equal strata, at
// a place of its own.
__device__ inline uint64_t sample_pos(uint32_t i, uint64_t n) {
  const uint64_t lo = (uint64_t)i * n / kLowSample, hi = (uint64_t)(i + 1) * n / kLowSample;
  uint32_t x = i * 0x9E3779B1u;
  x ^= x >> 15;
  x *= 0x85EBCA77u;
  x ^= x >> 13;
  return lo + (((hi - lo) * (uint64_t)(x >> 16)) >> 16);
}

// Lowest digit to sort by, from a sample of the n keys (ordered images in
// k[], thread t's item i at LowTile::pos): the largest low for which few keys
// are expected to agree with another one from bit 8 * low up, among those that
// leave out a digit that varies and leave an even number of varying ones (the
// result then lands where the keys were); 0 if none.  `even_only`: every digit
// from low up is a pass, so low itself is even.  The n / kLowSample keys
// between two neighbouring samples are taken as spread evenly over the gap
// between them; equal samples are taken as equal keys.  256 threads, all of
// them; every thread returns the answer.  About 9 us alone on the chip, of
// which the sample's reads are 2.
__device__ inline uint32_t choose_low(LowTile::Smem& sm, uint64_t (&k)[4], uint64_t n, bool even_only,
                                      uint32_t* s_sum) {
  const uint32_t tid = threadIdx.x;
  uint32_t none[1];
  LowTile t{sm, k, none, kLowSample, 4};
  if (tid < 8) s_sum[tid] = 0;
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
  const float per = (float)n * (4096.0f / (float)kLowSample);
  // Ties expected of this thread's four gaps at low = 0, in 1/4096 of a
  // sample; 256 times as many with every digit, up to the whole sample.
  float ties[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t p = tid + (uint32_t)j * 256;
    ties[j] = 0.0f;
    if (p + 1 < kLowSample) {
      // The staged samples are in order but for a few neighbours: those count
      // as close ones.
      const uint64_t a = sk[p], b = sk[p + 1];
      if (a != b) ties[j] = per * __builtin_amdgcn_rcpf(b > a ? (float)(b - a) : 1.0f);
    }
  }
#pragma unroll
  for (uint32_t low = 1; low < 8; ++low) {
    if (!((allowed >> low) & 1u)) continue;
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) sum += fminf(ties[j] * (float)(1ull << (8 * low)), 4096.0f);
    const uint32_t w = wave_incl_scan_dpp((uint32_t)sum);
    if ((tid & 63u) == 63u) atomicAdd(&s_sum[low], w);
  }
  lds_barrier();
  for (uint32_t low = 7; low > 0; --low)
    if (((allowed >> low) & 1u) && s_sum[low] <= 4096u * kLowSample / kTieFrac) return low;
  return 0;
}

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
  // Long runs: a bit for every 32 positions of every tile (zeroed), and the
  // list, each at least kShortRun + 1 keys (the slots segmented only).
  uint32_t* long_seen;
  uint64_t* long_start;
  uint32_t* long_slot;

  // They take the look-back words, which are done with by then: the bits
  // those of pass 0 (left out whenever the kernels have work, so still zero),
  // the list the following passes'.
  void use_status(void* status, size_t pass_bytes, uint64_t tiles, uint32_t pass_tile_keys) {
    long_seen = reinterpret_cast<uint32_t*>(status);
    char* list = reinterpret_cast<char*>(status) + pass_bytes;
    long_start = reinterpret_cast<uint64_t*>(list);
    long_slot = reinterpret_cast<uint32_t*>(list + tiles * (pass_tile_keys / (kShortRun + 1) + 1) * sizeof(uint64_t));
  }
};
// Per tile of at most 16384 keys: 16384 / 256 bytes of bits in the 1024 of a
// pass, and 497 list entries of 12 bytes in those of seven.
static_assert(16384 / 256 <= 1024 && (16384 / (kShortRun + 1) + 1) * 12 <= 7 * 1024, "long runs fit the look-back words");

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
// chunks of kTieChunk keys: the chunk is staged in LDS (all loads in flight
// together) and the positions of keys greater than the key after them in their
// run are gathered into a list, so that few of them cost one round of the
// workgroup and equal keys cost nothing.  The thread of a run's first listed
// position sorts the run.  A run that crosses the chunk's end belongs to the
// chunk it starts in and is sorted in global memory.  Where a run starts and
// ends depends only on bits that no step changes, so a run has one owner and
// reads of other owners' keys decide nothing about it.
constexpr uint32_t kTieChunk = 2048;

template <typename V, bool KV>
__device__ inline void sort_run_serial(uint64_t* keys, V* vals, uint64_t p, uint64_t seg1, uint64_t t, int s,
                                       const Xform<uint64_t>& xf) {
  uint32_t len = 2;
  while (p + len < seg1 && len <= kShortRun && (to_ordered(keys[p + len], xf) >> s) == t) ++len;
  if (len > kShortRun) return;
  for (uint32_t i = 1; i < len; ++i) {
    const uint64_t raw = keys[p + i];
    const uint64_t x = to_ordered(raw, xf);
    uint32_t at = i;
    while (at > 0 && to_ordered(keys[p + at - 1], xf) > x) --at;
    if (at == i) continue;
    V y{};
    if constexpr (KV) y = vals[p + i];
    for (uint32_t q = i; q > at; --q) {
      keys[p + q] = keys[p + q - 1];
      if constexpr (KV) vals[p + q] = vals[p + q - 1];
    }
    keys[p + at] = raw;
    if constexpr (KV) vals[p + at] = y;
  }
}

template <typename V, bool KV>
__global__ __launch_bounds__(256) void tie_fix_kernel(TieArgs<V> a) {
  constexpr int PER = kTieChunk / 256;
  __shared__ uint64_t s_k[kTieChunk + 2];  // keys from one before the chunk to one past it
  __shared__ uint16_t s_tie[kTieChunk];
  __shared__ uint32_t s_nties;
  const uint32_t low = a.ctrl->low();
  if (low == 0) return;
  const int s = 8 * (int)low;
  const uint32_t tid = threadIdx.x;
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
  for (uint64_t c0 = start; c0 < end; c0 += kTieChunk) {
    const uint32_t m = end - c0 < kTieChunk ? (uint32_t)(end - c0) : kTieChunk;
    uint64_t k[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      k[j] = keys[c0 + (i < m ? i : m - 1)];
    }
    if (tid == 0) s_nties = 0;
    // Past the segment's ends: a key of another run.
    if (tid == 64) s_k[0] = c0 > seg0 ? to_ordered(keys[c0 - 1], a.xf) : ~to_ordered(keys[c0], a.xf);
    if (tid == 128) s_k[m + 1] = c0 + m < seg1 ? to_ordered(keys[c0 + m], a.xf) : ~to_ordered(keys[c0 + m - 1], a.xf);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      if (i < m) s_k[i + 1] = to_ordered(k[j], a.xf);
    }
    lds_barrier();
    // Element i of the chunk sits at s_k[i + 1].
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t i = tid + (uint32_t)j * 256;
      if (i < m) {
        const uint64_t x = s_k[i + 1], y = s_k[i + 2];
        if (y < x && (y >> s) == (x >> s)) s_tie[atomicAdd(&s_nties, 1u)] = (uint16_t)i;
      }
    }
    lds_barrier();
    const uint32_t nties = s_nties;
    for (uint32_t j = tid; j < nties; j += 256) {
      const uint32_t i = s_tie[j];
      const uint64_t t = s_k[i + 1] >> s;
      // The run's first and last key in the chunk, kShortRun away at most,
      // and whether an earlier position of it is listed too.
      uint32_t b = i, e = i + 1;
      bool first = true;
      while (b > 0 && i - b <= kShortRun && (s_k[b] >> s) == t) {
        first &= s_k[b] <= s_k[b + 1];
        --b;
      }
      while (e + 1 < m && e - b <= kShortRun && (s_k[e + 2] >> s) == t) ++e;
      if (e - b < kShortRun) {
        if (e >= m || (b == 0 && (s_k[0] >> s) == t) || (e + 1 == m && (s_k[m + 1] >> s) == t)) {
          // It crosses an end of the chunk: sorted below or by the chunk before.
        } else if (e == b + 1) {
          const uint64_t lo = keys[c0 + b], hi = keys[c0 + e];
          V vl{}, vh{};
          if constexpr (KV) {
            vl = vals[c0 + b];
            vh = vals[c0 + e];
          }
          keys[c0 + b] = hi;
          keys[c0 + e] = lo;
          if constexpr (KV) {
            vals[c0 + b] = vh;
            vals[c0 + e] = vl;
          }
          continue;
        } else {
          if (first) sort_run_serial<V, KV>(keys, vals, c0 + b, seg1, t, s, a.xf);
          continue;
        }
      }
      // Is its run a long one?
      const uint64_t p = c0 + i;
      const uint64_t back = p - seg0 > kShortRun ? p - kShortRun : seg0;
      const uint64_t fwd = seg1 - p > kShortRun + 1 ? p + kShortRun + 1 : seg1;
      const uint64_t rb = first_at_least(keys, back, p, t, s, a.xf);
      const uint64_t re = first_at_least(keys, p + 1, fwd, t + 1, s, a.xf);
      if (re - rb <= kShortRun) continue;
      const uint64_t run = rb > back ? rb : first_at_least(keys, seg0, rb, t, s, a.xf);
      // Two runs longer than 32 never start in the same 32 positions.
      const uint64_t at = a.tile_seg ? (uint64_t)a.seg_first[slot] * a.tile_keys + (run - seg0) : run;
      const uint32_t bit = 1u << ((at >> 5) & 31u);
      if (atomicOr(&a.long_seen[at >> 10], bit) & bit) continue;
      const uint32_t n_long = atomicAdd(&a.ctrl->long_count, 1u);
      a.long_start[n_long] = run;
      if (a.tile_seg) a.long_slot[n_long] = slot;
    }
    // The run that crosses the chunk's end.
    if (tid == 255) {
      const uint64_t t = s_k[m] >> s;
      if ((s_k[m + 1] >> s) == t) {
        uint32_t b = m - 1;
        while (b > 0 && m - b <= kShortRun && (s_k[b] >> s) == t) --b;
        if ((s_k[b] >> s) != t) sort_run_serial<V, KV>(keys, vals, c0 + b, seg1, t, s, a.xf);
      }
    }
    __syncthreads();  // before the next chunk's first key is read and the list is reused
  }
}

// Sorts the listed runs, a workgroup a run: in LDS where the run fits a tile,
// else digit by digit below ctrl->low() through the other buffer, tile after
// tile (a histogram read, then every tile sorted by the digit in LDS and
// written behind the tiles before it).  Such a run is one the sample did not
// see coming: the workgroup moves about 1e9 keys a second and digit.
template <typename V, bool KV, int ITEMS>
__global__ __launch_bounds__(1024) void long_run_kernel(TieArgs<V> a) {
  using Tile = BlockRadix<uint64_t, V, KV, 1024, ITEMS, true>;
  using Part = BlockRadix<uint64_t, V, KV, 1024, 4, false>;
  __shared__ union {
    typename Tile::Smem tile;
    typename Part::Smem part;
  } sm;
  __shared__ uint64_t s_off[256];
  __shared__ uint64_t s_end;
  const uint32_t count = a.ctrl->long_count, low = a.ctrl->low();
  const uint32_t tid = threadIdx.x;
  const int s = 8 * (int)low;
  uint64_t* const keys = a.keys0;
  uint64_t* const other = a.keys1;
  V* const vals = a.vals0;
  V* const vother = a.vals1;
  for (uint32_t job = blockIdx.x; job < count; job += gridDim.x) {
    const uint64_t p0 = a.long_start[job];
    if (tid == 0) {
      const uint64_t seg1 = a.tile_seg ? a.seg_range[2 * a.long_slot[job] + 1] : a.n;
      s_end = first_at_least(keys, p0, seg1, (to_ordered(keys[p0], a.xf) >> s) + 1, s, a.xf);
    }
    __syncthreads();
    const uint64_t len = s_end - p0;
    if (len <= Tile::CAP) {
      uint64_t k[ITEMS];
      V v[KV ? ITEMS : 1];
      const uint32_t m = (uint32_t)len;
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
      continue;
    }
    const uint64_t* ki = keys + p0;
    uint64_t* ko = other + p0;
    const V* vi = vals + p0;
    V* vo = vother + p0;
    for (uint32_t d = 0; d < low; ++d) {
      if (tid < 256) s_off[tid] = 0;
      __syncthreads();
      for (uint64_t i = tid; i < len; i += 1024)
        atomicAdd(reinterpret_cast<unsigned long long*>(&s_off[digit_of(to_ordered(ki[i], a.xf), 8 * d)]), 1ull);
      __syncthreads();
      if (tid == 0) {
        uint64_t run = 0;
        for (int i = 0; i < 256; ++i) {
          const uint64_t c = s_off[i];
          s_off[i] = run;
          run += c;
        }
      }
      __syncthreads();
      for (uint64_t c0 = 0; c0 < len; c0 += Part::CAP) {
        const uint32_t m = len - c0 < Part::CAP ? (uint32_t)(len - c0) : Part::CAP;
        uint64_t k[4];
        V v[KV ? 4 : 1];
        Part t{sm.part, k, v, m, (m + 1023) / 1024};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t p = t.pos(i);
          const bool in = (uint32_t)i < t.items && p < m;
          k[i] = in ? to_ordered(ki[c0 + p], a.xf) : ~0ull;
          if constexpr (KV) v[i] = in ? vi[c0 + p] : V(0);
        }
        t.clear_masks();
        t.digit(8 * (int)d);
        // Wave 0's first slots are the digits' starts in the tile.
        const uint32_t* const first = t.counts();
        const uint64_t* const sk = t.keys();
        const V* const sv = t.vals();
        for (uint32_t p = tid; p < m; p += 1024) {
          const uint64_t x = sk[p];
          const uint32_t dg = digit_of(x, 8 * (int)d);
          const uint64_t dst = s_off[dg] + (p - first[dg]);
          ko[dst] = from_ordered(x, a.xf);
          if constexpr (KV) vo[dst] = sv[p];
        }
        __syncthreads();
        // Slots past the tile sit in the last digit.
        if (tid < 256) s_off[tid] += (tid == 255 ? m : first[tid + 1] < m ? first[tid + 1] : m) -
                                     (first[tid] < m ? first[tid] : m);
        __syncthreads();
      }
      const uint64_t* const kt = ki;
      ki = ko;
      ko = const_cast<uint64_t*>(kt);
      const V* const vt = vi;
      vi = vo;
      vo = const_cast<V*>(vt);
    }
    if (low & 1u) {
      for (uint64_t i = tid; i < len; i += 1024) {
        ko[i] = ki[i];
        if constexpr (KV) vo[i] = vi[i];
      }
      __syncthreads();
    }
  }
}

template <typename V, bool KV>
void launch_tie_fix(const TieArgs<V>& t, uint64_t tiles, uint64_t n_keys, hipStream_t stream, LaunchTimer* timer) {
  // Keys a thread of a run's tile: what fits the registers without spills.
  constexpr int ITEMS = !KV ? 12 : sizeof(V) == 4 ? 8 : 6;
  if (timer) timer->begin("tie_fix", n_keys * 8, stream);
  hipLaunchKernelGGL((tie_fix_kernel<V, KV>), dim3((uint32_t)tiles), dim3(256), 0, stream, t);
  hipLaunchKernelGGL((long_run_kernel<V, KV, ITEMS>), dim3((uint32_t)std::min<uint64_t>(256, n_keys / 16384 + 1)),
                     dim3(1024), 0, stream, t);
  if (timer) timer->end(stream);
}

}  // namespace gs
