// Stable radix sort of one tile held by one workgroup (LDS and registers),
// the core of the small-array and small-segment sorts (block_sort.hip).
//
// The tile is sorted by the bits that differ between its keys, not by the
// whole key: the highest two, three or four 8-bit digits of that range are
// sorted LSD in LDS, which orders all but a few neighbours.  The full keys are then
// checked, and on the way out a key that lies in a short run of keys equal in
// the sorted bits finds its place in it by comparing full keys with its
// neighbours.  Only a tile with a long run out of order (many keys that
// differ far below their highest differing bit) is sorted again over the
// whole range.
//
// What bounds it: latency, and LDS work for the largest tiles.  A digit costs
// five LDS operations a key for its rank (the lane-mask match of the onesweep
// passes), one for its slot and two (four with payloads) for the move, three
// barriers and one scan by a single wave (four digits a lane, the wave scan on
// DPP).
#pragma once

#include "gs_device.h"

namespace gs {

// Inclusive prefix sum over the wave on the DPP crossbar: six dependent VALU
// steps instead of six LDS permutes (rows of 16 by shifts of 1, 2, 4, 8, then
// the row totals by the two row broadcasts).  Every lane must be active.
__device__ inline uint32_t wave_incl_scan_dpp(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
  return x;
}

// OR over the wave, valid in lane 63.
__device__ inline uint32_t wave_or_dpp(uint32_t x) {
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
  return x;
}

// Longest run of keys equal in the sorted bits whose keys find their places
// by comparison (a key reads up to this many neighbours on each side).
constexpr uint32_t kFixRun = 8;
// Digits are added until random keys would leave at most this many pairs
// equal in them (m^2 / 2 over the slots): any such pair costs a second look at
// the whole tile, about half a digit, and more of them cost their comparisons.
constexpr uint32_t kTiePairs = 8;

// ALIAS: the ranking tables share the staging buffer (two more barriers a
// digit) where both would not fit the LDS or would halve the workgroups a CU
// holds.
template <typename U, typename V, bool KV, int THREADS, int ITEMS, bool ALIAS>
struct BlockRadix {
  static constexpr int WAVES = THREADS / kWave;
  static constexpr uint32_t CAP = THREADS * ITEMS;
  static constexpr size_t TABLES = (size_t)WAVES * 256 * 12;  // per wave: 256 lane masks, 256 counts
  static constexpr size_t STAGE = (size_t)CAP * (sizeof(U) + (KV ? sizeof(V) : 0));
  static constexpr size_t BYTES = ALIAS ? (TABLES > STAGE ? TABLES : STAGE) : TABLES + STAGE;

  struct Smem {
    alignas(16) unsigned char buf[BYTES];
    U red[WAVES][2];
    uint32_t seen[kWave];  // a byte per value of the highest digit
    uint32_t flag;
  };

  Smem& sm;
  U (&k)[ITEMS];
  V (&v)[KV ? ITEMS : 1];
  uint32_t m;      // keys of the tile
  uint32_t items;  // ceil(m / THREADS): item slots in use

  __device__ unsigned long long* masks() const {
    return reinterpret_cast<unsigned long long*>(sm.buf + (ALIAS ? 0 : STAGE)) + (threadIdx.x >> 6) * 256;
  }
  __device__ uint32_t* counts() const {
    return reinterpret_cast<uint32_t*>(sm.buf + (ALIAS ? 0 : STAGE) + (size_t)WAVES * 256 * 8);
  }
  __device__ U* keys() const { return reinterpret_cast<U*>(sm.buf); }
  __device__ V* vals() const { return reinterpret_cast<V*>(sm.buf + (size_t)CAP * sizeof(U)); }

  // Position of item i of this thread (wave-striped over the items in use,
  // so item order within a wave, then wave order, is tile order).
  __device__ uint32_t pos(int i) const {
    return (threadIdx.x >> 6) * (kWave * items) + (uint32_t)i * kWave + (threadIdx.x & 63u);
  }

  // The wave's own table rows before the first digit, and its counts before
  // every digit (the masks clear themselves).
  __device__ void clear_masks() const {
    uint4* p = reinterpret_cast<uint4*>(masks());
    for (uint32_t i = threadIdx.x & 63u; i < 128; i += kWave) p[i] = make_uint4(0, 0, 0, 0);
  }

  // One digit: bits [shift, shift + 8) of the keys, stably, registers ->
  // staging.  Slots past the tile (pos >= m) hold all-ones keys: they take
  // the digit's largest value and stay last.
  __device__ void digit(int shift) const {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (ALIAS) clear_masks();
    uint32_t* const cnt = counts();
    uint32_t* const wc = cnt + wave * 256;
    reinterpret_cast<uint4*>(wc)[lane] = make_uint4(0, 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    unsigned long long* const wm = masks();
    uint32_t r[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if ((uint32_t)i < items) {
        const uint32_t d = digit_of(k[i], shift);
        uint64_t peers;
        if (ballot(d != (uint32_t)__builtin_amdgcn_readfirstlane(d)) == 0) {
          peers = ~0ull;  // one digit in the whole wave: 64 lanes on one word would serialise
        } else {
          uint32_t* const half = reinterpret_cast<uint32_t*>(&wm[d]) + (lane >> 5);
          __hip_atomic_fetch_or(half, 1u << (lane & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          __builtin_amdgcn_wave_barrier();
          peers = __hip_atomic_load(&wm[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          __builtin_amdgcn_wave_barrier();
          __hip_atomic_store(half, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        const uint32_t old = wc[d];
        __builtin_amdgcn_wave_barrier();
        wc[d] = old + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        r[i] = old + count_below(peers);
      }
    }
    lds_barrier();
    // Wave 0: totals of four digits a lane, their exclusive starts, and
    // every wave's first slot of each digit, in place of its count
    // (read twice rather than held: the keys and ranks leave no registers
    // for 16 waves' counts).
    if (wave == 0) {
      uint4* const row = reinterpret_cast<uint4*>(cnt) + lane;
      uint4 t = make_uint4(0, 0, 0, 0);
#pragma unroll 4
      for (int w = 0; w < WAVES; ++w) {
        const uint4 c = row[w * 64];
        t.x += c.x;
        t.y += c.y;
        t.z += c.z;
        t.w += c.w;
      }
      const uint32_t sum = t.x + t.y + t.z + t.w;
      uint4 run;
      run.x = wave_incl_scan_dpp(sum) - sum;
      run.y = run.x + t.x;
      run.z = run.y + t.y;
      run.w = run.z + t.z;
#pragma unroll 4
      for (int w = 0; w < WAVES; ++w) {
        const uint4 c = row[w * 64];
        row[w * 64] = run;
        run.x += c.x;
        run.y += c.y;
        run.z += c.z;
        run.w += c.w;
      }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
      if ((uint32_t)i < items) r[i] += wc[digit_of(k[i], shift)];
    if (ALIAS) lds_barrier();  // the offsets are read before the staging overwrites them
    U* const sk = keys();
    V* const sv = vals();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if ((uint32_t)i < items) {
        sk[r[i]] = k[i];
        if constexpr (KV) sv[r[i]] = v[i];
      }
    }
    lds_barrier();
  }

  // Staging -> registers, in tile order.
  __device__ void read_back() const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if ((uint32_t)i < items) {
        k[i] = keys()[pos(i)];
        if constexpr (KV) v[i] = vals()[pos(i)];
      }
    }
    if (ALIAS) lds_barrier();  // every key is out before the tables are cleared
  }

  // The staged keys, sorted by their bits from s up: 0 if they are in order,
  // 1 if not, 3 if a key out of order lies in a run (keys equal from bit s up)
  // too long for one thread.
  __device__ uint32_t check(int s) const {
    const U* const sk = keys();
    bool bad = false, lng = false;
#pragma unroll 4
    for (uint32_t p = threadIdx.x; p + 1 < m; p += THREADS) {
      const U a = sk[p], b = sk[p + 1];
      if (b < a) {
        bad = true;
        const U t = a >> s;
        uint32_t len = 2;
        for (uint32_t q = p; q > 0 && len <= kFixRun && (U)(sk[q - 1] >> s) == t; --q) ++len;
        for (uint32_t q = p + 2; q < m && len <= kFixRun && (U)(sk[q] >> s) == t; ++q) ++len;
        lng |= len > kFixRun;
      }
    }
    if (bad)
      __hip_atomic_fetch_or(&sm.flag, lng ? 3u : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    lds_barrier();
    return sm.flag;
  }

  // Bits in which keys of the tile differ.
  __device__ U varying() const {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    U o = 0, z = 0;  // ones seen, zeros seen
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if ((uint32_t)i < items && pos(i) < m) {
        o |= k[i];
        z |= ~k[i];
      }
    }
    U ow = wave_or_dpp((uint32_t)o), zw = wave_or_dpp((uint32_t)z);
    if constexpr (sizeof(U) == 8) {
      ow |= (U)wave_or_dpp((uint32_t)(o >> 32)) << 32;
      zw |= (U)wave_or_dpp((uint32_t)(z >> 32)) << 32;
    }
    if (lane == 63) {
      sm.red[wave][0] = ow;
      sm.red[wave][1] = zw;
    }
    if (wave == 0) sm.seen[lane] = 0;
    if (threadIdx.x == 0) sm.flag = 0;
    lds_barrier();
    o = z = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      o |= sm.red[w][0];
      z |= sm.red[w][1];
    }
    return o & z;
  }

  // Values of the eight bits below and at hb among the first item of every
  // thread (a sample of at least m / items keys).
  __device__ uint32_t top_values(int hb) const {
    const int sh = hb > 7 ? hb - 7 : 0;
    if (pos(0) < m) reinterpret_cast<unsigned char*>(sm.seen)[digit_of(k[0], sh)] = 1;
    lds_barrier();
    const uint32_t c = wave_incl_scan_dpp((uint32_t)__popc(sm.seen[threadIdx.x & 63u]));
    return (uint32_t)__builtin_amdgcn_readlane((int)c, 63);
  }

  // Sorts the tile held in registers (ordered images at pos(i); all ones past
  // m) into the staging arrays.  Returns kInOrder if every key is equal (the
  // staging is not written), kSorted, or the bit s >= 0 from which up the
  // staged keys are sorted: place() then gives each key its place.
  static constexpr int kInOrder = -2, kSorted = -1;
  __device__ int sort() const {
    const U diff = varying();
    if (diff == 0) return kInOrder;
    if (!ALIAS) clear_masks();
    const int hb = (int)sizeof(U) * 8 - 1 - (sizeof(U) == 8 ? __clzll((long long)diff) : __clz((int)diff));
    const int lb = sizeof(U) == 8 ? __ffsll((long long)diff) - 1 : __ffs((int)diff) - 1;
    const int all = (hb - lb + 8) / 8;
    // Two digits hold about 256 slots for each value of the highest one that
    // occurs, and each further one 256 times as many.
    int top = 2;
    for (uint64_t slots = (uint64_t)top_values(hb) * 256; top < all && (uint64_t)m * m > 2 * kTiePairs * slots;
         slots *= 256)
      ++top;
    bool whole = all <= top;
    const int s = whole ? lb : hb + 1 - 8 * top;
    int d = s, end = s + 8 * (whole ? all : top);
    // One loop over the digits, entered again where a tile needs its whole
    // range (one copy of the digit's code).
    for (;;) {
      digit(d);
      d += 8;
      if (d >= end) {
        if (whole) return kSorted;
        const uint32_t f = check(s);
        if (f == 0) return kSorted;
        if (!(f & 2u)) return s;
        whole = true;
        d = lb;
        end = lb + 8 * all;
      }
      read_back();
    }
  }

  // Place of the staged key x at p in the run of keys that agree with it from
  // bit s up (at most kFixRun keys, or in order already): stable.
  __device__ uint32_t place(uint32_t p, U x, int s) const {
    const U* const sk = keys();
    const U t = x >> s;
    uint32_t dst = p;
    const uint32_t lo = p > kFixRun ? p - kFixRun : 0, hi = p + kFixRun < m ? p + kFixRun : m - 1;
    for (uint32_t q = p; q > lo; --q) {
      const U y = sk[q - 1];
      if ((U)(y >> s) != t) break;
      dst -= y > x ? 1u : 0u;
    }
    for (uint32_t q = p + 1; q <= hi; ++q) {
      const U y = sk[q];
      if ((U)(y >> s) != t) break;
      dst += y < x ? 1u : 0u;
    }
    return dst;
  }

  // Hands every staged element to put(place, key, index in the staging); s is
  // what sort() returned.  Where neighbours may have to change places, four
  // keys and their neighbours are read together and only waves that hold a
  // tie look further.
  template <typename Put>
  __device__ void write_out(int s, Put put) const {
    const U* const sk = keys();
    if (s < 0) {
      for (uint32_t p = threadIdx.x; p < m; p += THREADS) put(p, sk[p], p);
      return;
    }
    for (uint32_t p0 = threadIdx.x; p0 < m; p0 += 4 * THREADS) {
      U x[4], a[4], b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t p = p0 + (uint32_t)j * THREADS, c = p < m ? p : m - 1;
        x[j] = sk[c];
        a[j] = sk[c ? c - 1 : 0];
        b[j] = sk[c + 1 < m ? c + 1 : c];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t p = p0 + (uint32_t)j * THREADS;
        if (p < m) {
          const U t = x[j] >> s;
          const bool tie = (p > 0 && (U)(a[j] >> s) == t) || (p + 1 < m && (U)(b[j] >> s) == t);
          put(tie ? place(p, x[j], s) : p, x[j], p);
        }
      }
    }
  }
};

}  // namespace gs
