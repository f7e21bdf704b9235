// Sorts of small arrays and small segments, one workgroup each: the tile is
// read once, sorted in LDS and registers (block_radix.h) and written once.
//
// Serves the same seam as the radix passes (thrust::sort / thrust::sort_by_key,
// src/cuda_utils.cu:424, :477) when n is at most one tile.  Stable: payloads
// ride along with their keys through every digit.
#include "block_radix.h"
#include "gs_internal.h"

namespace gs {

template <typename U, typename V, bool KV, int THREADS, int ITEMS, bool ALIAS>
__global__ __launch_bounds__(THREADS) void block_sort_kernel(U* __restrict__ keys, V* __restrict__ vals,
                                                             const uint64_t* __restrict__ seg_off,
                                                             const uint32_t* __restrict__ seg_ids, uint32_t n_single,
                                                             Xform<U> xf) {
  using Tile = BlockRadix<U, V, KV, THREADS, ITEMS, ALIAS>;
  __shared__ typename Tile::Smem sm;
  uint64_t lo = 0;
  uint32_t m = n_single;
  if (seg_off != nullptr) {
    const uint32_t seg = seg_ids ? seg_ids[blockIdx.x] : blockIdx.x;
    lo = seg_off[seg];
    m = (uint32_t)(seg_off[seg + 1] - lo);
  }
  if (m <= 1 || m > Tile::CAP) return;
  U k[ITEMS];
  V v[KV ? ITEMS : 1];
  Tile t{sm, k, v, m, (m + THREADS - 1) / THREADS};
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t p = t.pos(i);
    const bool in = (uint32_t)i < t.items && p < m;
    k[i] = in ? keys[lo + p] : U(0);
    if constexpr (KV) v[i] = in ? vals[lo + p] : V(0);
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) k[i] = ((uint32_t)i < t.items && t.pos(i) < m) ? to_ordered(k[i], xf) : U(~U(0));
  const int s = t.sort();
  if (s == Tile::kInOrder) return;
  const V* const sv = t.vals();
  t.write_out(s, [&](uint32_t dst, U x, uint32_t p) {
    keys[lo + dst] = from_ordered(x, xf);
    if constexpr (KV) vals[lo + dst] = sv[p];
  });
}

// Measured (kernel alone, u32 + u32, against the bitonic network it replaced):
// 1000 pairs 6.4 us (21.8); 20,000 lognormal arrays' segments of up to 4096
// pairs 0.17 ms (0.72).  Batches of equal arrays, whole call: 108 Gkeys/s at
// 4096 keys, 114 at 8000 (two 512-thread workgroups a CU), 83 at 16000 (one).
// A single array is sorted here up to the widest tile: 16384 u32 pairs 40 us,
// 4096 12 us, where the radix passes take 60-70 us at these sizes.
//
// Tile geometries by length: one wave up to 256 keys (no barrier waits on
// another wave), 256 x 4 up to 1024, 512 x 8 (a single array, alone on the
// chip: 1024 x 4) up to 4096, then 512 threads (two workgroups a CU) and 1024
// with as many keys a thread as stage in the 160 KB of LDS, up to 16.
constexpr uint32_t kClassLen[3] = {256, 1024, 4096};

static constexpr int wide_items(int kb, int vb) {
  return kb + vb <= 8 ? 16 : kb + vb == 12 ? 12 : 9;
}


uint32_t block_sort_max(int kb, int vb) {
  const int w = kb + vb;
  return w == 4 ? 8192 : (w == 8) ? 4096 : 2048;
}

uint32_t block_sort_tile_max(int kb, int vb) { return 1024u * (uint32_t)wide_items(kb, vb); }

uint32_t block_sort_class_len(int kb, int vb, int cls) {
  return cls < 3 ? kClassLen[cls] : 512u * (uint32_t)wide_items(kb, vb);
}

int block_sort_class(int kb, int vb, uint32_t len) {
  for (int c = 0; c < kBlockClasses - 1; ++c)
    if (len <= block_sort_class_len(kb, vb, c)) return c;
  return kBlockClasses - 1;
}

template <int VB>
struct BValT {
  using T = uint32_t;
};
template <>
struct BValT<8> {
  using T = uint64_t;
};

template <typename U, int VB>
static hipError_t launch_block_sort(void* keys, void* vals, const uint64_t* d_off, const uint32_t* d_ids,
                                    uint32_t nblocks, uint32_t n, const XformParams& xp, hipStream_t stream, int cls) {
  using V = typename BValT<VB>::T;
  constexpr bool KV = VB != 0;
  constexpr int W = wide_items(sizeof(U), VB);
  constexpr bool BIG = sizeof(U) + VB > 8;  // 4096 such elements beside the tables leave one workgroup a CU
  const Xform<U> xf{(U)xp.float_mask, (U)xp.sign_flip, (U)xp.desc_mask};
  U* k = reinterpret_cast<U*>(keys);
  V* v = reinterpret_cast<V*>(vals);
  if (cls == 0)
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 64, 4, false>), dim3(nblocks), dim3(64), 0, stream, k, v, d_off,
                       d_ids, n, xf);
  else if (cls == 1)
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 256, 4, false>), dim3(nblocks), dim3(256), 0, stream, k, v, d_off,
                       d_ids, n, xf);
  else if (cls == 2 && d_off != nullptr)
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 512, 8, BIG>), dim3(nblocks), dim3(512), 0, stream, k, v, d_off,
                       d_ids, n, xf);
  else if (cls == 2)
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 1024, 4, false>), dim3(nblocks), dim3(1024), 0, stream, k, v,
                       d_off, d_ids, n, xf);
  else if (cls == 3)
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 512, W, true>), dim3(nblocks), dim3(512), 0, stream, k, v, d_off,
                       d_ids, n, xf);
  else
    hipLaunchKernelGGL((block_sort_kernel<U, V, KV, 1024, W, true>), dim3(nblocks), dim3(1024), 0, stream, k, v, d_off,
                       d_ids, n, xf);
  return hipGetLastError();
}

static hipError_t dispatch_block_sort(int kb, int vb, void* keys, void* vals, const uint64_t* d_off,
                                      const uint32_t* d_ids, uint32_t nblocks, uint32_t n, const XformParams& xf,
                                      hipStream_t stream, int cls) {
  if (kb == 4) {
    if (vb == 0) return launch_block_sort<uint32_t, 0>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
    if (vb == 4) return launch_block_sort<uint32_t, 4>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
    if (vb == 8) return launch_block_sort<uint32_t, 8>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
  } else if (kb == 8) {
    if (vb == 0) return launch_block_sort<uint64_t, 0>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
    if (vb == 4) return launch_block_sort<uint64_t, 4>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
    if (vb == 8) return launch_block_sort<uint64_t, 8>(keys, vals, d_off, d_ids, nblocks, n, xf, stream, cls);
  }
  return hipErrorInvalidValue;
}

hipError_t block_sort(int kb, int vb, void* keys, void* vals, uint32_t n, const XformParams& xf, hipStream_t stream) {
  if (n > block_sort_tile_max(kb, vb)) return hipErrorInvalidValue;
  if (n <= 1) return hipSuccess;
  return dispatch_block_sort(kb, vb, keys, vals, nullptr, nullptr, 1, n, xf, stream, block_sort_class(kb, vb, n));
}

hipError_t block_sort_segments(int kb, int vb, void* keys, void* vals, const uint64_t* d_offsets,
                               const uint32_t* d_seg_ids, uint32_t nblocks, const XformParams& xf, hipStream_t stream,
                               int cls) {
  if (nblocks == 0) return hipSuccess;
  if (cls < 0 || cls >= kBlockClasses) return hipErrorInvalidValue;
  return dispatch_block_sort(kb, vb, keys, vals, d_offsets, d_seg_ids, nblocks, 0, xf, stream, cls);
}

}  // namespace gs
