// dst[i] = src[idx[i]] for large sources in random order, bucket first.
//
// A direct gather of random indexes fetches a cache line of 128 bytes from
// memory for every element, whatever its width.  Here the indexes are first
// put in order of source region, tile by tile, so that every region is pulled
// through one XCD's L2 while all of its readers run:
//   split  a tile of kTile indexes a workgroup: sorted in LDS by region (in
//          any order within one), written as 32-bit index and 16-bit place in
//          the tile, with a row of region starts
//   pull   region after region, the regions dealt to the XCDs: the elements
//          of every tile's indexes of the region, to the tile's part of dst
//   place  every tile of dst put in order of place through LDS
//
// Nothing crosses a tile but the pull's reads of src, so there is no
// histogram, scan or look-back.  Where the indexes are better gathered directly
// (direct_is_better) the split kernel leaves, the pull's workgroups gather and the
// place kernel leaves.  An index of 2^32 or more is split as what it is below
// that, an element of the source too, and gathered again by the place kernel;
// where dst lies over idx such a tile is gathered directly, at the end.
//
// What bounds it: the pull, at about 1 ms for 2^27 elements the rate of L2
// accesses (one an element); then split and place, bytes (14 and, with u32, 10
// an element).  Measured, 2^27 random indexes: u16 2.58 -> 1.31 ms, u32 2.56 ->
// 1.53, u64 3.27 -> 2.09; 2^24: u32 0.314 -> 0.205, u64 0.337 -> 0.269.
// In-order indexes cost the leaving kernels' 10 us (2^24 u32: 38 -> 48 us, 2^25
// 97 -> 108); below 2^24 elements that weighs more than the saving (2^23 u32: 144
// -> 108, u8 88 -> 96), so kGatherSplitMin lies there.  Gathering in the split
// kernel instead leaves one kernel less, but its large workgroups lose the lines
// that neighbours share (2^24 u32 shuffled within 64 K elements: 122 -> 176 us).
#include <algorithm>

#include "block_radix.h"
#include "gs_device.h"
#include "gs_internal.h"

namespace gs {

namespace {

constexpr uint32_t kThreads = 1024;
constexpr int kItems = 16;
constexpr uint32_t kTile = kThreads * kItems;
constexpr uint32_t kMinRegions = 256, kMaxRegions = 512;
constexpr uint32_t kRow = kMaxRegions + 8;  // region starts of a tile, and where the last one ends
constexpr uint32_t kXcds = 8;

// Bytes of source a region holds at most, if the indexes are below n (half of
// an XCD's L2), and regions there are at least.
constexpr uint64_t kRegionBytes = 2u << 20;
// Whether the indexes are best gathered directly, from 16 pairs of neighbours
// spread over the array: over a third of them are so close that they find each
// other's lines in the L2, or all indexes lie in so little of src that caches
// hold most of it (against the split, random indexes over 8 MB cost 10 ps an
// element, over 32 MB 17; the split 12 and, with 8-byte elements, 18), or they
// lie in so much of it that hardly two of them share a line: a quarter of them
// are `far` or more.  Every wave of every workgroup finds the same answer.
constexpr uint32_t kNearBytes = 256u << 10;
__device__ inline bool direct_is_better(const uint64_t* idx, uint64_t n, uint32_t elem_bytes, uint64_t far) {
  const uint32_t lane = threadIdx.x & 31u;
  const uint64_t a = idx[(n - 1) / 16 * (lane >> 1) + (lane & 1u)];
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)a, 0xB1, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(a >> 32), 0xB1, 0xf, 0xf, false);
  const uint64_t b = ((uint64_t)hi << 32) | lo;
  const uint64_t small = (elem_bytes == 8 ? 48u << 20 : 14u << 20) / elem_bytes;
  return __popcll(ballot((a < b ? b - a : a - b) < kNearBytes / elem_bytes)) >= 24 ||  // a pair counts four times
         ballot(a >= small) == 0 || __popcll(ballot(a >= far)) >= 16;                  // an index twice
}

// Three quarters of the elements of a source in which n random indexes fall on a
// line of 128 bytes 0.8 times each, below 2^25 indexes 1.5 times: past that the
// split costs more than it saves (2^24 indexes: u32 over 16 times as many elements
// 364 us directly and 349 split, over 32 times 404 and 425; u64 over 4 times 339
// and 337, over 16 times 432 and 466; 2^25: u64 over 16 times as many 948 and 911,
// over 24 times 968 and 986).  At most 2^32, where a split index ends.
uint64_t far_index(uint64_t n, uint32_t elem_bytes) {
  return std::min<uint64_t>(n * (n < (1ull << 25) ? 64 : 120) / elem_bytes, 1ull << 32);
}

// Where a tile's slots start in its part of ent, place and dst.  Tiles are
// 64 KB apart there, so without it the pulls of one region, at about one slot
// in every tile, would all meet in a few memory channels.
__device__ inline uint32_t slot_shift(uint32_t tile, uint32_t valid) {
  return valid == kTile ? (tile * 0x9E3779B1u) >> 18 : 0u;
}
static_assert(kTile == 1u << 14, "slot_shift gives 14 bits");

// What bounds it: the read of the indexes and the writes (14 bytes an element;
// 2^27 of them 0.36 ms, 5.2 TB/s), two workgroups a CU overlapping their phases.
// `apart`: dst does not lie over idx.
__global__ __launch_bounds__(kThreads, 8) void gather_split_kernel(const uint64_t* __restrict__ idx, uint64_t n,
                                                                   uint32_t elem_bytes, uint64_t far, bool apart,
                                                                   uint32_t shift, uint32_t regions,
                                                                   uint32_t* __restrict__ split,
                                                                   uint32_t* __restrict__ tickets,
                                                                   uint32_t* __restrict__ ent,
                                                                   uint16_t* __restrict__ place,
                                                                   uint16_t* __restrict__ rows) {
  __shared__ uint32_t s_cnt[kMaxRegions];
  __shared__ uint32_t s_buf[kTile];
  const uint32_t tid = threadIdx.x, tile = blockIdx.x;
  const bool direct = direct_is_better(idx, n, elem_bytes, far);
  if (tile == 0) {
    if (tid == 0) *split = !direct;
    if (tid < kXcds) tickets[tid * 32] = 0;
  }
  if (direct) return;
  const uint64_t base = (uint64_t)tile * kTile;
  const uint32_t valid = n - base < kTile ? (uint32_t)(n - base) : kTile;
  // Compiled twice, for whole tiles (no compares) and for the last one.
  auto tile_body = [&](auto full_tag) {
    constexpr bool full = decltype(full_tag)::value;
    const uint64_t* const ti = idx + base;
    for (uint32_t i = tid; i < kMaxRegions; i += kThreads) s_cnt[i] = 0;
    uint32_t x[kItems];
    uint32_t wide = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint64_t v =
          full ? (ti + j * (int)kThreads)[tid] : ti[min((uint32_t)j * kThreads + tid, valid - 1)];
      wide |= (uint32_t)(v >> 32);
      x[j] = (uint32_t)v;
    }
    uint16_t* const row = rows + (uint64_t)tile * kRow;
    const bool any_wide = __syncthreads_or(wide != 0);
    if (any_wide && !apart) {
      for (uint32_t i = tid; i < kRow; i += kThreads) row[i] = 0;
      return;
    }
    if (tid == 0) row[regions + 1] = any_wide;
    const uint32_t skew = slot_shift(tile, valid);
    auto region = [&](uint32_t v) { return (v >> shift) & (regions - 1); };
    uint32_t r[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t p = (uint32_t)j * kThreads + tid;
      r[j] = full || p < valid ? atomicAdd(&s_cnt[region(x[j])], 1u) : 0u;
    }
    lds_barrier();
    if (tid < kWave) {  // one wave: starts of the regions
      constexpr uint32_t PER = kMaxRegions / kWave / 4;
      uint4* const c = reinterpret_cast<uint4*>(s_cnt) + PER * tid;
      uint4 a[PER];
      uint32_t sum = 0;
#pragma unroll
      for (uint32_t i = 0; i < PER; ++i) {
        a[i] = c[i];
        sum += a[i].x + a[i].y + a[i].z + a[i].w;
      }
      uint32_t at = wave_incl_scan_dpp(sum) - sum;
#pragma unroll
      for (uint32_t i = 0; i < PER; ++i) {
        const uint4 y = make_uint4(at, at + a[i].x, at + a[i].x + a[i].y, at + a[i].x + a[i].y + a[i].z);
        at = y.w + a[i].w;
        c[i] = y;
      }
    }
    lds_barrier();
    for (uint32_t i = tid; i <= regions; i += kThreads) row[i] = (uint16_t)(i < regions ? s_cnt[i] : valid);
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      r[j] = (r[j] + s_cnt[region(x[j])] + skew) % kTile;
      if (full || (uint32_t)j * kThreads + tid < valid) s_buf[r[j]] = x[j];
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t p = (uint32_t)j * kThreads + tid;
      if (full || p < valid) (ent + base + j * (int)kThreads)[tid] = s_buf[p];
    }
    lds_barrier();
    uint16_t* const s_place = reinterpret_cast<uint16_t*>(s_buf);
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t p = (uint32_t)j * kThreads + tid;
      if (full || p < valid) s_place[r[j]] = (uint16_t)p;
    }
    lds_barrier();
    // The last tile's pairs past its end stay within the tile's part of place.
    uint32_t* const pw = reinterpret_cast<uint32_t*>(place + base);
#pragma unroll
    for (int j = 0; j < kItems / 2; ++j) {
      const uint32_t p = (uint32_t)j * kThreads + tid;
      if (full || 2 * p < valid) pw[p] = s_buf[p];
    }
  };
  if (valid == kTile)
    tile_body(std::true_type{});
  else
    tile_body(std::false_type{});
}

// Sixteen lanes a tile: a tile holds about 64 indexes of a region at 2^27
// elements (32 of 8-byte ones).
constexpr uint32_t kPullThreads = 256, kPullLanes = 16, kPullTiles = kPullThreads / kPullLanes;
constexpr int kPullUnroll = 8;
// Workgroups of the pull an XCD: three a CU.  More of them spread over more
// regions at a time and lose lines (2^27 u32 elements, a gather: 8 a CU 1.91
// ms, 4 a CU 1.74, 3 a CU 1.71, 2 a CU 1.75).  Dealing the jobs by ticket rather
// than by stride keeps them to one region or two: 2.46 -> 1.91.
constexpr uint32_t kPullGroups = 96;
// Workgroups launched, all of which gather where the tiles were not split (one
// launch less than with a kernel of its own).
constexpr uint32_t kPullGrid = 8192;

template <typename T>
__global__ __launch_bounds__(kPullThreads) void gather_pull_kernel(const T* __restrict__ src, const uint64_t* idx,
                                                                   T* dst, uint64_t n, uint32_t regions,
                                                                   const uint32_t* __restrict__ split,
                                                                   uint32_t* __restrict__ tickets,
                                                                   const uint32_t* __restrict__ ent,
                                                                   const uint16_t* __restrict__ rows) {
  if (!*split) {
    const uint64_t stride = (uint64_t)gridDim.x * kPullThreads;
    for (uint64_t i = (uint64_t)blockIdx.x * kPullThreads + threadIdx.x; i < n; i += stride) dst[i] = src[idx[i]];
    return;
  }
  constexpr uint32_t kWorkgroups = kXcds * kPullGroups;
  if (blockIdx.x >= kWorkgroups) return;
  constexpr int UN = kPullUnroll;
  const uint32_t tiles = (uint32_t)((n + kTile - 1) / kTile);
  const uint32_t xcd = blockIdx.x % kXcds;
  const uint32_t chunks = (tiles + kPullTiles - 1) / kPullTiles;
  const uint32_t jobs = regions / kXcds * chunks;
  const uint32_t group = threadIdx.x / kPullLanes, lane = threadIdx.x % kPullLanes;
  __shared__ uint32_t s_job[2];
  auto pull = [&](uint32_t b, uint32_t tile) {
    const uint16_t* const row = rows + (uint64_t)tile * kRow + b;
    const uint32_t end = row[1];
    const uint32_t skew = slot_shift(tile, (uint64_t)(tile + 1) * kTile <= n ? kTile : 0u);
    const uint32_t* const te = ent + (uint64_t)tile * kTile;
    T* const td = dst + (uint64_t)tile * kTile;
    for (uint32_t i = row[0] + lane; i < end; i += UN * kPullLanes) {
      uint32_t x[UN];
      T v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const uint32_t q = i + (uint32_t)u * kPullLanes;
        if (q < end) x[u] = __builtin_nontemporal_load(&te[(q + skew) % kTile]);
      }
#pragma unroll
      for (int u = 0; u < UN; ++u)
        if (i + (uint32_t)u * kPullLanes < end) v[u] = src[x[u]];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const uint32_t q = i + (uint32_t)u * kPullLanes;
        if (q < end) td[(q + skew) % kTile] = v[u];
      }
    }
  };
  // The first job is the workgroup's own, the next ones come from the XCD's
  // ticket, taken a job ahead.
  uint32_t job = blockIdx.x / kXcds;
  for (uint32_t turn = 0; job < jobs; turn ^= 1) {
    uint32_t next = 0;
    if (threadIdx.x == 0) next = kPullGroups + atomicAdd(&tickets[xcd * 32], 1u);
    const uint32_t b = xcd + kXcds * (job / chunks), tile = job % chunks * kPullTiles + group;
    if (tile < tiles) pull(b, tile);
    if (threadIdx.x == 0) s_job[turn] = next;
    lds_barrier();
    job = s_job[turn];
  }
}

// Two workgroups a CU but for 8-byte elements: at most 64 registers, which the
// addresses stay within where the items' offsets are uniform (89 registers, one
// workgroup: 0.39 ms for 2^27 u32 elements; 64: 0.25).
template <typename T>
__global__ __launch_bounds__(kThreads, sizeof(T) == 8 ? 4 : 8) void gather_place_kernel(
    const T* __restrict__ src, const uint64_t* idx, T* dst, uint64_t n, bool apart, uint32_t regions,
    const uint32_t* __restrict__ split, const uint16_t* __restrict__ place, const uint16_t* __restrict__ rows) {
  __shared__ T s_val[kTile];
  if (!*split) return;
  const uint32_t tid = threadIdx.x, tiles = (uint32_t)((n + kTile - 1) / kTile);
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint64_t base = (uint64_t)tile * kTile;
    T* const td = dst + base;
    const uint16_t* const row = rows + (uint64_t)tile * kRow + regions;
    const uint32_t valid = row[0];
    if (valid == 0) {  // not split, dst lies over idx
#pragma unroll 4
      for (uint64_t p = base + tid; p < n && p < base + kTile; p += kThreads) dst[p] = src[idx[p]];
      continue;
    }
    const bool wide = row[1] != 0;
    const uint16_t* const tp = place + (uint64_t)tile * kTile;
    uint16_t at[kItems];
    T v[kItems];
    if (valid == kTile) {
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        at[j] = (tp + j * (int)kThreads)[tid];
        v[j] = (td + j * (int)kThreads)[tid];
      }
    } else {
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const uint32_t p = min((uint32_t)j * kThreads + tid, valid - 1);
        at[j] = tp[p];
        v[j] = td[p];
      }
    }
    // Past the end of the last tile: its last element once more.
#pragma unroll
    for (int j = 0; j < kItems; ++j) s_val[at[j]] = v[j];
    lds_barrier();
    if (valid == kTile) {
#pragma unroll
      for (int j = 0; j < kItems; ++j) (td + j * (int)kThreads)[tid] = s_val[(uint32_t)j * kThreads + tid];
    } else {
      for (uint32_t p = tid; p < valid; p += kThreads) td[p] = s_val[p];
    }
    lds_barrier();
    if (wide)
#pragma unroll 4
      for (uint32_t p = tid; p < valid; p += kThreads) {
        const uint64_t x = idx[base + p];
        if (x >> 32) td[p] = src[x];
      }
  }
}

struct GatherLayout {
  uint64_t tiles;
  size_t off_ent, off_place, off_rows, total;
};

GatherLayout gather_layout(uint64_t n) {
  GatherLayout L{};
  L.tiles = (n + kTile - 1) / kTile;
  size_t o = 256 + kXcds * 128;  // whether the tiles were split; tickets, a line each
  L.off_ent = o;
  o += L.tiles * kTile * sizeof(uint32_t);
  L.off_place = o;
  o += L.tiles * kTile * sizeof(uint16_t);
  L.off_rows = o;
  o += align_up(L.tiles * kRow * sizeof(uint16_t), 256);
  L.total = o;
  return L;
}

template <typename T>
hipError_t gather_split_t(const T* src, const uint64_t* idx, T* dst, uint64_t n, unsigned char* ws,
                          hipStream_t stream) {
  const GatherLayout L = gather_layout(n);
  uint32_t* split = reinterpret_cast<uint32_t*>(ws);
  uint32_t* tickets = reinterpret_cast<uint32_t*>(ws + 256);
  uint32_t* ent = reinterpret_cast<uint32_t*>(ws + L.off_ent);
  uint16_t* place = reinterpret_cast<uint16_t*>(ws + L.off_place);
  uint16_t* rows = reinterpret_cast<uint16_t*>(ws + L.off_rows);
  const uint32_t tiles = (uint32_t)L.tiles;
  const uint32_t regions = n * sizeof(T) > kMinRegions * kRegionBytes ? kMaxRegions : kMinRegions;
  uint32_t shift = 0;
  while (((n - 1) >> shift) >= regions) ++shift;
  const uintptr_t di = reinterpret_cast<uintptr_t>(dst), ii = reinterpret_cast<uintptr_t>(idx);
  const bool apart = di + n * sizeof(T) <= ii || ii + n * sizeof(uint64_t) <= di;
  hipLaunchKernelGGL(gather_split_kernel, dim3(tiles), dim3(kThreads), 0, stream, idx, n, (uint32_t)sizeof(T),
                     far_index(n, sizeof(T)), apart, shift, regions, split, tickets, ent, place, rows);
  hipLaunchKernelGGL(gather_pull_kernel<T>, dim3(kPullGrid), dim3(kPullThreads), 0, stream, src, idx, dst, n, regions,
                     split, tickets, ent, rows);
  hipLaunchKernelGGL(gather_place_kernel<T>, dim3(std::min(tiles, 512u)), dim3(kThreads), 0, stream, src, idx, dst, n,
                     apart, regions, split, place, rows);
  return hipGetLastError();
}

}  // namespace

size_t gather_split_bytes(int elem_bytes, uint64_t n) {
  if (n < kGatherSplitMin || n >= (1ull << 40)) return 0;
  return gather_layout(n).total;
}

hipError_t gather_split(int elem_bytes, const void* src, const uint64_t* idx, void* dst, uint64_t n, void* workspace,
                        hipStream_t stream) {
  unsigned char* ws = reinterpret_cast<unsigned char*>(workspace);
  switch (elem_bytes) {
    case 1:
      return gather_split_t(reinterpret_cast<const uint8_t*>(src), idx, reinterpret_cast<uint8_t*>(dst), n, ws,
                            stream);
    case 2:
      return gather_split_t(reinterpret_cast<const uint16_t*>(src), idx, reinterpret_cast<uint16_t*>(dst), n, ws,
                            stream);
    case 4:
      return gather_split_t(reinterpret_cast<const uint32_t*>(src), idx, reinterpret_cast<uint32_t*>(dst), n, ws,
                            stream);
    case 8:
      return gather_split_t(reinterpret_cast<const uint64_t*>(src), idx, reinterpret_cast<uint64_t*>(dst), n, ws,
                            stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace gs
