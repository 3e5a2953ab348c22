// Uniform-grid cell list for gfx950.
//
// Replaces the reference's grid build (src/optixNSearch/sort.cpp:34-136,
// 500-627; grid.cu:13-31,213-329): integer bbox via atomics, meta-grid Morton
// cell ids, atomicAdd local indices (non-deterministic within a cell),
// Thrust scan and sort.  Here:
//   bbox        float min/max, block reduction (no atomics on 6 addresses);
//   cell_keys   raster cell id per point (x fastest), or the level-0 Morton
//               code of a hierarchical grid (morton_keys);
//   radix sort  stable sort of (cell, index) -> points ordered by (cell, index);
//   cell_bounds cell_start[c] = first sorted position with key >= c: one
//               binary search per 4096-cell tile, then each tile's cells
//               searched inside its own key range staged in LDS, so the work
//               per thread is bounded however many cells are empty; a Morton
//               level l uses key >> 3l and the same sorted keys;
//   gather      sorted points as float4 (x, y, z, bits(original index)) so one
//               16-byte load yields a candidate and its output index.
// Query order: Morton code of the query's cell (helper_mortonCode.h:19-34
// restated), radix-sorted, so a wave's queries walk neighbouring cells.
#include <float.h>

#include <algorithm>

#include "common.h"
#include "internal.h"

namespace rtnn {

constexpr int kBboxThreads = 256;

__device__ inline void wave_minmax(float& mn, float& mx) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
  }
}

template <int TH = kBboxThreads>
__device__ inline void block_bbox(float v[6], float* sh /*6 * waves*/) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  constexpr int nw = TH / kWave;
#pragma unroll
  for (int a = 0; a < 3; ++a) wave_minmax(v[a], v[a + 3]);
  if (lane == 0)
#pragma unroll
    for (int a = 0; a < 6; ++a) sh[a * nw + w] = v[a];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int a = 0; a < 3; ++a) {
      float mn = sh[a * nw], mx = sh[(a + 3) * nw];
      for (int i = 1; i < nw; ++i) {
        mn = fminf(mn, sh[a * nw + i]);
        mx = fmaxf(mx, sh[(a + 3) * nw + i]);
      }
      v[a] = mn;
      v[a + 3] = mx;
    }
  }
}

__device__ inline void accum_point(float x, float y, float z, float v[6], uint32_t& bad) {
  if (!(isfinite(x) && isfinite(y) && isfinite(z))) {
    ++bad;
    return;
  }
  v[0] = fminf(v[0], x); v[1] = fminf(v[1], y); v[2] = fminf(v[2], z);
  v[3] = fmaxf(v[3], x); v[4] = fmaxf(v[4], y); v[5] = fmaxf(v[5], z);
}
__device__ inline void accum_point(const float* xyz, uint64_t i, float v[6], uint32_t& bad) {
  accum_point(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], v, bad);
}
// Four points held by three 16-byte words.
__device__ inline void accum_quad(const float4& a, const float4& b, const float4& c, float v[6],
                                  uint32_t& bad) {
  accum_point(a.x, a.y, a.z, v, bad);
  accum_point(a.w, b.x, b.y, v, bad);
  accum_point(b.z, b.w, c.x, v, bad);
  accum_point(c.y, c.z, c.w, v, bad);
}

// Box and non-finite count of n points, and with COPY their copy into dst, in
// one launch.  At small n the launches, not the bytes, are the cost: 1500 points
// set and searched take 56 us, 92 us when a copy, a clear, two reductions and a
// copy back of the box did this (100,000 points: 108 and 143 us; the kernel
// itself 6 and 7 us).  The last block to finish folds the blocks' partial boxes: they are stored past the XCDs' own
// L2s, and are there (vmcnt 0) before the block takes its ticket.  *ticket is
// zero before and after.  VEC: src (and dst) are 16-byte aligned.
template <bool COPY, bool VEC>
__global__ __launch_bounds__(kBboxThreads) void k_bbox(const float* __restrict__ src,
                                                       float* __restrict__ dst, uint64_t n,
                                                       float* __restrict__ part,
                                                       uint32_t* __restrict__ ticket,
                                                       float* __restrict__ out,
                                                       uint32_t* __restrict__ nonfinite) {
  __shared__ float sh[6 * kBboxThreads / kWave];
  __shared__ uint32_t s_bad, s_last;
  float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  uint32_t bad = 0;
  if (threadIdx.x == 0) s_bad = 0;
  __syncthreads();
  const uint64_t t0 = (uint64_t)blockIdx.x * kBboxThreads + threadIdx.x;
  const uint64_t nt = (uint64_t)gridDim.x * kBboxThreads;
  uint64_t done = 0;
  if constexpr (VEC) {
    const float4* s4 = reinterpret_cast<const float4*>(src);
    float4* d4 = reinterpret_cast<float4*>(dst);
    for (uint64_t i = t0; i < n / 4; i += nt) {
      const float4 a = s4[3 * i], b = s4[3 * i + 1], c = s4[3 * i + 2];
      if constexpr (COPY) {
        d4[3 * i] = a;
        d4[3 * i + 1] = b;
        d4[3 * i + 2] = c;
      }
      accum_quad(a, b, c, v, bad);
    }
    done = n / 4 * 4;
  }
  for (uint64_t i = done + t0; i < n; i += nt) {
    const float x = src[3 * i], y = src[3 * i + 1], z = src[3 * i + 2];
    if constexpr (COPY) {
      dst[3 * i] = x;
      dst[3 * i + 1] = y;
      dst[3 * i + 2] = z;
    }
    accum_point(x, y, z, v, bad);
  }
  if (bad) atomicAdd(&s_bad, bad);
  block_bbox(v, sh);
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int a = 0; a < 6; ++a)
      __hip_atomic_store(&part[8 * blockIdx.x + a], v[a], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(reinterpret_cast<uint32_t*>(part) + 8 * blockIdx.x + 6, s_bad,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             gridDim.x - 1;
    s_bad = 0;
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  for (int a = 0; a < 3; ++a) {
    v[a] = FLT_MAX;
    v[a + 3] = -FLT_MAX;
  }
  bad = 0;
  for (uint32_t i = threadIdx.x; i < gridDim.x; i += kBboxThreads) {
    float p[6];
    for (int a = 0; a < 6; ++a)
      p[a] = __hip_atomic_load(&part[8 * i + a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bad += __hip_atomic_load(reinterpret_cast<uint32_t*>(part) + 8 * i + 6, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    for (int a = 0; a < 3; ++a) {
      v[a] = fminf(v[a], p[a]);
      v[a + 3] = fmaxf(v[a + 3], p[a + 3]);
    }
  }
  if (bad) atomicAdd(&s_bad, bad);
  block_bbox(v, sh);
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int a = 0; a < 6; ++a) out[a] = v[a];
    *nonfinite = s_bad;
    __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

hipError_t bbox(const float* src, float* dst, uint64_t n, float* part, uint32_t* ticket,
                float* out, uint32_t* nonfinite, hipStream_t st) {
  const uint64_t want = (n + kBboxThreads * 4 - 1) / (kBboxThreads * 4);
  const dim3 nb((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(want, kBboxBlocks)));
  const dim3 th(kBboxThreads);
  const bool vec = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
  if (dst && vec)
    hipLaunchKernelGGL((k_bbox<true, true>), nb, th, 0, st, src, dst, n, part, ticket, out, nonfinite);
  else if (dst)
    hipLaunchKernelGGL((k_bbox<true, false>), nb, th, 0, st, src, dst, n, part, ticket, out, nonfinite);
  else if (vec)
    hipLaunchKernelGGL((k_bbox<false, true>), nb, th, 0, st, src, dst, n, part, ticket, out, nonfinite);
  else
    hipLaunchKernelGGL((k_bbox<false, false>), nb, th, 0, st, src, dst, n, part, ticket, out, nonfinite);
  return hipGetLastError();
}

// One block of TH threads per cloud.  What bounds it is how many loads the block
// of the largest cloud keeps in flight: each thread takes four points (three
// 16-byte words) at a time from the first multiple of four points on, and clouds
// of 4096 points or more on average get 1024 threads (1024 clouds of up to
// 200,000 points, 38 million in all: 280 us, 410 with 256 threads, 466 with 256 that
// take a point at a time; blocks of small clouds would sit idle in 1024).
// VEC: xyz is 16-byte aligned.
constexpr uint64_t kBboxWideCloud = 4096;

template <bool VEC, int TH>
__global__ __launch_bounds__(TH) void k_bbox_seg(const float* __restrict__ xyz,
                                                 const uint64_t* __restrict__ off,
                                                 float* __restrict__ out,
                                                 uint32_t* __restrict__ nonfinite) {
  __shared__ float sh[6 * TH / kWave];
  const uint32_t c = blockIdx.x;
  float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  uint32_t bad = 0;
  const uint64_t i0 = off[c], i1 = off[c + 1];
  uint64_t head = i1, rest = i1;  // points before the first quad, after the last
  if constexpr (VEC) {
    const float4* x4 = reinterpret_cast<const float4*>(xyz);
    head = std::min<uint64_t>(i1, (i0 + 3) & ~3ull);
    rest = std::max<uint64_t>(head, i1 & ~3ull);
#pragma unroll 2
    for (uint64_t j = head / 4 + threadIdx.x; j < rest / 4; j += TH)
      accum_quad(x4[3 * j], x4[3 * j + 1], x4[3 * j + 2], v, bad);
  }
  for (uint64_t i = i0 + threadIdx.x; i < head; i += TH) accum_point(xyz, i, v, bad);
  for (uint64_t i = rest + threadIdx.x; i < i1; i += TH) accum_point(xyz, i, v, bad);
  if (bad) atomicAdd(nonfinite, bad);
  block_bbox<TH>(v, sh);
  if (threadIdx.x == 0)
    for (int a = 0; a < 6; ++a) out[6 * c + a] = v[a];
}

hipError_t bbox_segmented(const float* xyz, const uint64_t* offsets, uint32_t nclouds,
                          uint64_t n, float* out, uint32_t* nonfinite, hipStream_t st) {
  if (nclouds == 0) return hipSuccess;
  const bool vec = (reinterpret_cast<uintptr_t>(xyz) & 15) == 0;
  auto launch = [&](auto kernel, int th) {
    hipLaunchKernelGGL(kernel, dim3(nclouds), dim3(th), 0, st, xyz, offsets, out, nonfinite);
  };
  if (n / nclouds >= kBboxWideCloud)
    vec ? launch(k_bbox_seg<true, 1024>, 1024) : launch(k_bbox_seg<false, 1024>, 1024);
  else
    vec ? launch(k_bbox_seg<true, 256>, 256) : launch(k_bbox_seg<false, 256>, 256);
  return hipGetLastError();
}

// ---- device-side planning of the batched grids (no host round trip, so the
// whole batched pipeline can be captured in a graph).

__device__ inline uint64_t cells_sat(int d0, int d1, int d2) {
  const double c = (double)d0 * (double)d1 * (double)d2;
  return c > 1e15 ? (uint64_t)1e15 : (uint64_t)d0 * (uint64_t)d1 * (uint64_t)d2;
}

// Dims of one cloud's grid; the host planner's arithmetic (-ffp-contract=off).
__device__ inline void plan_dims(const float* bb, float inv, bool empty, int d[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float e = (bb[a + 3] - bb[a]) * inv;
    const float f = floorf(e) + 1.0f;
    d[a] = empty ? 1 : (int)fminf(fmaxf(f, 1.0f), 2.0e9f);  // NaN, -inf -> 1
  }
}

constexpr int kPlanThreads = 1024;

__device__ inline uint64_t block_sum_u64(uint64_t v, uint64_t* sh) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  __syncthreads();
  if (lane == 0) sh[w] = v;
  __syncthreads();
  uint64_t t = 0;
  for (int i = 0; i < kPlanThreads / kWave; ++i) t += sh[i];
  return t;
}

// One block.  Grows the edge by 1.25x until the total cell count fits cap
// (the host planner's loop), then writes every cloud's GridDesc with its
// cell_base.  If no edge fits within 200 steps, every cloud gets a single
// cell (inv = 0): slow but exact, and status[1] is set.
__global__ __launch_bounds__(kPlanThreads) void k_plan_batched(
    const float* __restrict__ bboxes, const uint64_t* __restrict__ off, uint32_t nclouds,
    float cell, const float* __restrict__ cells, uint64_t cap, GridDesc* __restrict__ grids,
    uint32_t* __restrict__ status) {
  __shared__ uint64_t sh[kPlanThreads / kWave];
  __shared__ uint64_t s_scan[kPlanThreads];
  // Cloud i's edge: cells[i] (size classes) or cell, times the common growth.
  float gf = 1.0f;
  bool ok = false;
  for (int tries = 0; tries <= 200 && !ok; ++tries) {
    uint64_t tot = 0;
    for (uint32_t i = threadIdx.x; i < nclouds; i += kPlanThreads) {
      int d[3];
      plan_dims(bboxes + 6 * i, 1.0f / ((cells ? cells[i] : cell) * gf), off[i + 1] == off[i], d);
      tot = min(tot + cells_sat(d[0], d[1], d[2]), (uint64_t)1e15);  // no wrap
    }
    tot = block_sum_u64(tot, sh);
    ok = tot <= cap && tot < 0xfffffff0ull;
    if (!ok) gf *= 1.25f;
  }
  if (!ok && threadIdx.x == 0) status[1] = 1u;
  uint64_t carry = 0;
  for (uint32_t i0 = 0; i0 < nclouds; i0 += kPlanThreads) {
    const uint32_t i = i0 + threadIdx.x;
    int d[3] = {1, 1, 1};
    bool empty = true;
    float c = FLT_MAX, inv = 0.0f;
    if (i < nclouds) {
      empty = off[i + 1] == off[i];
      if (ok) {
        c = (cells ? cells[i] : cell) * gf;
        inv = 1.0f / c;
        plan_dims(bboxes + 6 * i, inv, empty, d);
      }
    }
    const uint64_t mine = i < nclouds ? cells_sat(d[0], d[1], d[2]) : 0;
    // inclusive scan of this chunk (Hillis-Steele in LDS)
    __syncthreads();
    s_scan[threadIdx.x] = mine;
    __syncthreads();
    for (int o = 1; o < kPlanThreads; o <<= 1) {
      const uint64_t t = threadIdx.x >= (uint32_t)o ? s_scan[threadIdx.x - o] : 0;
      __syncthreads();
      s_scan[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nclouds) {
      GridDesc g;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        g.mn[a] = empty ? 0.0f : bboxes[6 * i + a];
        g.dim[a] = d[a];
      }
      g.inv = inv;
      g.cell = c;
      g.cell_base = (uint32_t)(carry + s_scan[threadIdx.x] - mine);
      g.point_base = (uint32_t)off[i];
      g.npoints = (uint32_t)(off[i + 1] - off[i]);
      g.morton = 0;
      grids[i] = g;
    }
    carry += s_scan[kPlanThreads - 1];
  }
  if (threadIdx.x == 0) status[2] = (uint32_t)carry;
}

hipError_t plan_batched(const float* bboxes, const uint64_t* offsets, uint32_t nclouds,
                        float cell, const float* cells, uint64_t cap, GridDesc* grids,
                        uint32_t* status, hipStream_t st) {
  if (nclouds == 0) return hipSuccess;
  hipLaunchKernelGGL(k_plan_batched, dim3(1), dim3(kPlanThreads), 0, st, bboxes, offsets,
                     nclouds, cell, cells, cap, grids, status);
  return hipGetLastError();
}

__device__ inline int cell_of(float x, float mn, float inv, int dim) {
  float c = floorf((x - mn) * inv);
  c = fminf(fmaxf(c, 0.0f), (float)(dim - 1));
  return (int)c;
}

__device__ inline uint32_t find_cloud(const uint64_t* off, uint32_t nclouds, uint64_t i) {
  // last c with off[c] <= i
  uint32_t lo = 0, hi = nclouds - 1;
  while (lo < hi) {
    uint32_t m = (lo + hi + 1) >> 1;
    if (off[m] <= i) lo = m; else hi = m - 1;
  }
  return lo;
}

__global__ __launch_bounds__(256) void k_cell_keys(const float* __restrict__ xyz, uint64_t n,
                                                   const GridDesc* __restrict__ grids,
                                                   const uint64_t* __restrict__ off,
                                                   uint32_t nclouds,
                                                   uint32_t* __restrict__ keys,
                                                   uint32_t* __restrict__ vals,
                                                   uint32_t* __restrict__ counts) {
  // The block's first cloud by one binary search; a thread steps forward from
  // it (clouds are contiguous, so a block of 256 points spans few of them).
  __shared__ uint32_t s_c0;
  const uint64_t i0 = (uint64_t)blockIdx.x * 256;
  const uint64_t i = i0 + threadIdx.x;
  if (threadIdx.x == 0) s_c0 = nclouds > 1 ? find_cloud(off, nclouds, i0) : 0u;
  __syncthreads();
  if (i >= n) return;
  uint32_t c = s_c0;
  while (c + 1 < nclouds && off[c + 1] <= i) ++c;
  const GridDesc g = grids[c];
  int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
  int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
  int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
  uint32_t key = g.cell_base + ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) *
                                   (uint32_t)g.dim[0] + (uint32_t)cx;
  keys[i] = key;
  vals[i] = (uint32_t)i;
  if (counts) atomicAdd(&counts[key], 1u);
}

hipError_t cell_keys(const float* xyz, uint64_t n, const GridDesc* grids,
                     const uint64_t* offsets, uint32_t nclouds, uint32_t* keys,
                     uint32_t* vals, uint32_t* counts, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_keys, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, n,
                     grids, offsets, nclouds, keys, vals, counts);
  return hipGetLastError();
}

// One cloud: the grid descriptor comes by value (no host-to-device copy before
// the first kernel) and thread 0 stores it to gstore for the kernels after it.
__global__ __launch_bounds__(256) void k_cell_keys1(const float* __restrict__ xyz, uint64_t n,
                                                    const GridDesc g, GridDesc* __restrict__ gstore,
                                                    uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ vals) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0) *gstore = g;
  if (i >= n) return;
  const int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
  const int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
  const int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
  keys[i] = g.morton ? hilbert3((uint32_t)cx, (uint32_t)cy, (uint32_t)cz)
                     : g.cell_base + ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) *
                                         (uint32_t)g.dim[0] + (uint32_t)cx;
  vals[i] = (uint32_t)i;
}

hipError_t cell_keys_single(const float* xyz, uint64_t n, const GridDesc& g, GridDesc* gstore,
                            uint32_t* keys, uint32_t* vals, hipStream_t st) {
  const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, (n + 255) / 256);
  hipLaunchKernelGGL(k_cell_keys1, dim3(blocks), dim3(256), 0, st, xyz, n, g, gstore, keys, vals);
  return hipGetLastError();
}

// cell_start[c] = first sorted position whose key (>> shift) is >= c, for c
// in [0, ncells] (entry ncells holds n), so a cell's points are
// [cell_start[c], cell_start[c+1]) and no counts, atomics or scan are needed.
// The cells are cut into tiles: k_tile_bounds finds each tile's first sorted
// position by binary search (one thread per tile), then one block per tile
// writes its cells, each a lower_bound over the tile's keys staged in LDS.
// Every block writes exactly one tile, however the points are spread (empty
// space costs the same as occupied space).  Tiles hold 4096 cells, fewer for
// small tables (down to 256) so that at least ~1024 blocks share the work:
// a 125k-cell table in 31 blocks of 4096 left most CUs idle.
constexpr uint32_t kCellTileMax = 4096;
constexpr uint32_t kCellTileMin = 256;
constexpr uint32_t kCellTileKeys = 4096;  // keys staged in LDS per tile

uint32_t cell_tile(uint64_t ncells1) {
  uint32_t t = kCellTileMax;
  while (t > kCellTileMin && ncells1 / t < 1024) t >>= 1;
  return t;
}

__device__ inline uint64_t lower_bound_shifted(const uint32_t* __restrict__ keys, uint64_t lo,
                                               uint64_t hi, uint64_t c, int shift) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if ((uint64_t)(keys[mid] >> shift) < c) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(256) void k_tile_bounds(const uint32_t* __restrict__ keys, uint64_t n,
                                                     uint64_t ncells1, uint32_t ntiles,
                                                     uint32_t tile, int shift,
                                                     uint64_t* __restrict__ tb) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t > ntiles) return;
  const uint64_t c = min((uint64_t)t * tile, ncells1);
  tb[t] = lower_bound_shifted(keys, 0, n, c, shift);
}

__global__ __launch_bounds__(256) void k_cell_fill(const uint32_t* __restrict__ keys,
                                                   uint64_t ncells1, uint32_t tile, int shift,
                                                   const uint64_t* __restrict__ tb,
                                                   uint32_t* __restrict__ cs) {
  __shared__ uint32_t s_keys[kCellTileKeys];
  const uint32_t t = blockIdx.x;
  const uint64_t c0 = (uint64_t)t * tile;
  const uint64_t j0 = tb[t], j1 = tb[t + 1];
  const uint64_t m = j1 - j0;
  const bool staged = m <= kCellTileKeys;
  if (staged)
    for (uint32_t i = threadIdx.x; i < m; i += 256) s_keys[i] = keys[j0 + i] >> shift;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < tile; i += 256) {
    const uint64_t c = c0 + i;
    if (c >= ncells1) break;
    uint64_t pos;
    if (staged) {
      uint32_t lo = 0, hi = (uint32_t)m;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if ((uint64_t)s_keys[mid] < c) lo = mid + 1; else hi = mid;
      }
      pos = j0 + lo;
    } else {
      pos = lower_bound_shifted(keys, j0, j1, c, shift);
    }
    cs[c] = (uint32_t)pos;
  }
}

uint64_t cell_bounds_tmp_words(uint64_t ncells) {
  const uint32_t tile = cell_tile(ncells + 1);
  return 2 * ((ncells + 1 + tile - 1) / tile + 1) + 2;
}

hipError_t cell_bounds(const uint32_t* sorted_keys, uint64_t n, uint32_t ncells,
                       uint32_t* cell_start, uint32_t* tmp, hipStream_t st, int shift) {
  const uint64_t ncells1 = (uint64_t)ncells + 1;
  const uint32_t tile = cell_tile(ncells1);
  const uint32_t ntiles = (uint32_t)((ncells1 + tile - 1) / tile);
  uint64_t* tb = reinterpret_cast<uint64_t*>(tmp);
  hipLaunchKernelGGL(k_tile_bounds, dim3((ntiles + 1 + 255) / 256), dim3(256), 0, st,
                     sorted_keys, n, ncells1, ntiles, tile, shift, tb);
  hipLaunchKernelGGL(k_cell_fill, dim3(ntiles), dim3(256), 0, st, sorted_keys, ncells1, tile,
                     shift, tb, cell_start);
  return hipGetLastError();
}

// ---- raster grids by counting
//
// The order of the points inside a cell decides no result (rows are ordered by
// (d2, index)), so a raster grid needs no sort: every point takes a rank in its
// cell from an atomic counter, the counters are scanned into cell_start, and
// each point is written to cell_start[cell] + rank.  Three or four launches
// where the stable sort takes ten or more (keys, three per radix pass, cell
// table, gather): 100k uniform points, 15625 cells: 46 -> 22 us on the device,
// and 5 us less of the host per launch.

// Rank of this lane's point in its cell.  Points of a wave that share the cell
// of its first or its last one (clouds stored cell by cell, many points in one
// place) are added with one atomic, the rest one by one.
constexpr int kShareMin = 8;
__device__ inline uint32_t cell_rank(uint32_t* __restrict__ counts, uint32_t key, bool valid) {
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t rank = 0;
  bool todo = valid;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint64_t left = __ballot(todo);
    if (left == 0) return rank;
    const int lead = i == 0 ? __ffsll((unsigned long long)left) - 1 : 63 - __clzll((long long)left);
    const uint32_t k0 = (uint32_t)__builtin_amdgcn_readlane((int)key, lead);
    const uint64_t same = __ballot(todo && key == k0);
    if (__popcll(same) < kShareMin) continue;
    uint32_t base = 0;
    if (lane == lead) base = atomicAdd(&counts[k0], (uint32_t)__popcll(same));
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, lead);
    if (todo && key == k0) {
      rank = base + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
      todo = false;
    }
  }
  if (todo) rank = atomicAdd(&counts[key], 1u);
  return rank;
}

// One cloud: the descriptor by value, stored to gstore for the kernels after.
__global__ __launch_bounds__(256) void k_cell_count1(const float* __restrict__ xyz, uint64_t n,
                                                     const GridDesc g,
                                                     GridDesc* __restrict__ gstore,
                                                     uint32_t* __restrict__ counts,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ ranks) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0) *gstore = g;
  const bool valid = i < n;
  uint32_t key = 0;
  if (valid) {
    const int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
    const int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
    const int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
    key = ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] + (uint32_t)cx;
  }
  const uint32_t rank = cell_rank(counts, key, valid);
  if (valid) {
    keys[i] = key;
    ranks[i] = rank;
  }
}

// Clouds packed back to back, grids[c] for cloud c.
__global__ __launch_bounds__(256) void k_cell_count(const float* __restrict__ xyz, uint64_t n,
                                                    const GridDesc* __restrict__ grids,
                                                    const uint64_t* __restrict__ off,
                                                    uint32_t nclouds,
                                                    uint32_t* __restrict__ counts,
                                                    uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ ranks) {
  __shared__ uint32_t s_c0;
  const uint64_t i0 = (uint64_t)blockIdx.x * 256;
  const uint64_t i = i0 + threadIdx.x;
  if (threadIdx.x == 0) s_c0 = nclouds > 1 ? find_cloud(off, nclouds, i0) : 0u;
  __syncthreads();
  const bool valid = i < n;
  uint32_t key = 0;
  if (valid) {
    uint32_t c = s_c0;
    while (c + 1 < nclouds && off[c + 1] <= i) ++c;
    const GridDesc g = grids[c];
    const int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
    const int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
    const int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
    key = g.cell_base + ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] +
          (uint32_t)cx;
  }
  const uint32_t rank = cell_rank(counts, key, valid);
  if (valid) {
    keys[i] = key;
    ranks[i] = rank;
  }
}

// Exclusive scan of the cell counters into cell_start (ncells + 1 entries, the
// last the point count), leaving the counters at zero for the next build (a
// store only where they were not).  A block scans kScanCells cells; `part`
// holds the cells' sums per block, or is null when one block takes them all
// (looped over tables of up to kOneBlockCells cells: one launch).
constexpr int kCellScanThreads = 1024;
constexpr uint32_t kScanCells = kCellScanThreads * 4;
constexpr uint32_t kOneBlockCells = 16 * kScanCells;

// Four counters of this thread, cells c .. c + 3.
__device__ inline uint4 load_counts(const uint32_t* __restrict__ counts, uint64_t c,
                                    uint64_t ncells) {
  if (c + 4 <= ncells) return *reinterpret_cast<const uint4*>(counts + c);
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (c < ncells) v.x = counts[c];
  if (c + 1 < ncells) v.y = counts[c + 1];
  if (c + 2 < ncells) v.z = counts[c + 2];
  return v;
}

__device__ inline uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__global__ __launch_bounds__(kCellScanThreads) void k_cell_sums(
    const uint32_t* __restrict__ counts, uint64_t ncells, uint32_t* __restrict__ part) {
  __shared__ uint32_t sh[kCellScanThreads / kWave];
  const uint64_t c = (uint64_t)blockIdx.x * kScanCells + 4ull * threadIdx.x;
  const uint4 v = load_counts(counts, c, ncells);
  const uint32_t s = wave_sum(v.x + v.y + v.z + v.w);
  if (threadIdx.x % kWave == 0) sh[threadIdx.x / kWave] = s;
  __syncthreads();
  if (threadIdx.x < kWave) {
    const uint32_t t = wave_sum(threadIdx.x < kCellScanThreads / kWave ? sh[threadIdx.x] : 0u);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kCellScanThreads) void k_cell_scan(uint32_t* __restrict__ counts,
                                                                uint64_t ncells, uint64_t n,
                                                                const uint32_t* __restrict__ part,
                                                                uint32_t* __restrict__ cell_start) {
  constexpr int nw = kCellScanThreads / kWave;
  __shared__ uint32_t sh[nw];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  uint32_t run = 0;
  if (part) {  // points in the blocks before this one
    uint32_t s = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kCellScanThreads) s += part[b];
    s = wave_sum(s);
    if (lane == 0) sh[w] = s;
    __syncthreads();
    for (int i = 0; i < nw; ++i) run += sh[i];
    __syncthreads();
  }
  const uint64_t first = part ? (uint64_t)blockIdx.x * kScanCells : 0;
  const uint64_t last = part ? min(first + kScanCells, ncells) : ncells;
  for (uint64_t c0 = first; c0 < last; c0 += kScanCells) {
    const uint64_t c = c0 + 4ull * threadIdx.x;
    const uint4 v = load_counts(counts, c, ncells);
    const uint32_t own = v.x + v.y + v.z + v.w;
    uint32_t incl = own;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t t = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) sh[w] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < nw; ++i) {
      const uint32_t t = sh[i];
      before += i < w ? t : 0u;
      total += t;
    }
    const uint32_t s = run + before + incl - own;
    const uint4 o = make_uint4(s, s + v.x, s + v.x + v.y, s + v.x + v.y + v.z);
    if (c + 4 <= ncells) {
      *reinterpret_cast<uint4*>(cell_start + c) = o;
      if (own) *reinterpret_cast<uint4*>(counts + c) = make_uint4(0u, 0u, 0u, 0u);
    } else {
      const uint32_t ov[3] = {o.x, o.y, o.z};
      for (int i = 0; i < 3; ++i)
        if (c + i < ncells) {
          cell_start[c + i] = ov[i];
          counts[c + i] = 0u;
        }
    }
    run += total;
    __syncthreads();  // sh is written again
  }
  if (threadIdx.x == 0 && last == ncells) cell_start[ncells] = (uint32_t)n;
}

// Points to their places: reads in input order, 16-byte stores.
__global__ __launch_bounds__(256) void k_cell_place(const float* __restrict__ xyz,
                                                    const uint32_t* __restrict__ keys,
                                                    const uint32_t* __restrict__ ranks, uint64_t n,
                                                    const uint32_t* __restrict__ cell_start,
                                                    float4* __restrict__ spts) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t pos = cell_start[keys[i]] + ranks[i];
  spts[pos] = make_float4(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2],
                          __uint_as_float((uint32_t)i));
}

uint64_t cell_scan_tmp_words(uint64_t ncells) {
  return ncells <= kOneBlockCells ? 1 : (ncells + kScanCells - 1) / kScanCells;
}

hipError_t cell_scan_place(const float* xyz, uint64_t n, uint64_t ncells, uint32_t* counts,
                                  const uint32_t* keys, const uint32_t* ranks,
                                  uint32_t* cell_start, uint32_t* tmp, float4* spts,
                                  hipStream_t st) {
  if (ncells <= kOneBlockCells) {
    hipLaunchKernelGGL(k_cell_scan, dim3(1), dim3(kCellScanThreads), 0, st, counts, ncells, n,
                       (const uint32_t*)nullptr, cell_start);
  } else {
    const dim3 grid((uint32_t)((ncells + kScanCells - 1) / kScanCells));
    hipLaunchKernelGGL(k_cell_sums, grid, dim3(kCellScanThreads), 0, st, counts, ncells, tmp);
    hipLaunchKernelGGL(k_cell_scan, grid, dim3(kCellScanThreads), 0, st, counts, ncells, n, tmp,
                       cell_start);
  }
  hipLaunchKernelGGL(k_cell_place, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, keys,
                     ranks, n, cell_start, spts);
  return hipGetLastError();
}

hipError_t cell_count_single(const float* xyz, uint64_t n, const GridDesc& g, GridDesc* gstore,
                             uint32_t* counts, uint32_t* keys, uint32_t* ranks, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_count1, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, n, g,
                     gstore, counts, keys, ranks);
  return hipGetLastError();
}

// How the points are spread over the cells of grid g, from m of them (all, or
// draws with replacement): each adds one to its cell's counter, hashed into a
// table of 2^tbits where that is the smaller, and takes the number of points
// counted there before it as its rank.  *spread becomes the sums over the draws
// of rank and of rank (rank - 1) / 2: the pairs and the triples of draws that
// share a cell; then spread->done is 1.  Random atomics bound it, hence the sample
// (131,072 draws 10 us, a million points 60); folded by the last block to finish,
// as in k_bbox.
__global__ __launch_bounds__(256) void k_cell_spread(const float* __restrict__ xyz, uint64_t n,
                                                     uint32_t m, const GridDesc g, bool hashed,
                                                     int tbits, uint32_t* __restrict__ table,
                                                     unsigned long long* __restrict__ part,
                                                     uint32_t* __restrict__ ticket,
                                                     CellSpread* __restrict__ spread) {
  __shared__ unsigned long long s_sum[2];
  __shared__ uint32_t s_last;
  const int lane = threadIdx.x & (kWave - 1);
  if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t d = blockIdx.x * 256 + threadIdx.x;
  const bool valid = d < m;
  uint32_t key = 0;
  if (valid) {
    uint64_t i = d;
    if (m < n) {  // Steele, Lea and Flood's mixing function (SplitMix64, 2014)
      uint64_t z = (d + 1ull) * 0x9e3779b97f4a7c15ull;
      z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
      z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
      i = ((z >> 32) * n) >> 32;
    }
    const int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
    const int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
    const int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
    key = ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] + (uint32_t)cx;
    if (hashed) key = (key * 0x9e3779b1u) >> (32 - tbits);  // Knuth's multiplicative hash
  }
  const uint64_t rank = cell_rank(table, key, valid);
  unsigned long long v[2] = {rank, rank * (rank - (rank ? 1 : 0)) / 2};
  auto fold = [&]() {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) v[c] += __shfl_xor(v[c], o, kWave);
      if (lane == 0 && v[c]) atomicAdd(&s_sum[c], v[c]);
    }
    __syncthreads();
  };
  fold();
  if (threadIdx.x == 0) {
    for (int c = 0; c < 2; ++c) {
      __hip_atomic_store(&part[2 * blockIdx.x + c], s_sum[c], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      s_sum[c] = 0;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             gridDim.x - 1;
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  v[0] = v[1] = 0;
  for (uint32_t b = threadIdx.x; b < gridDim.x; b += 256)
    for (int c = 0; c < 2; ++c)
      v[c] += __hip_atomic_load(&part[2 * b + c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  fold();
  if (threadIdx.x == 0) {
    __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    spread->pairs = s_sum[0];
    spread->triples = s_sum[1];
    __hip_atomic_store(&spread->done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

hipError_t cell_spread(const float* xyz, uint64_t n, uint32_t m, const GridDesc& g, bool hashed,
                       int tbits, uint32_t* table, uint64_t* part, uint32_t* ticket,
                       CellSpread* spread, hipStream_t st) {
  if (m == 0 || m > kSpreadDraws || m > n || tbits < 1 || tbits > 31) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_cell_spread, dim3((m + 255) / 256), dim3(256), 0, st, xyz, n, m, g, hashed,
                     tbits, table, reinterpret_cast<unsigned long long*>(part), ticket, spread);
  return hipGetLastError();
}

hipError_t cell_count(const float* xyz, uint64_t n, const GridDesc* grids,
                      const uint64_t* offsets, uint32_t nclouds, uint32_t* counts, uint32_t* keys,
                      uint32_t* ranks, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_count, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, n,
                     grids, offsets, nclouds, counts, keys, ranks);
  return hipGetLastError();
}

// Level-0 Morton key of each point's cell on grid g (cubic, 2^bits cells per
// axis); the sort by this key makes every coarser level's cells contiguous.
__global__ __launch_bounds__(256) void k_morton_keys(const float* __restrict__ xyz, uint64_t n,
                                                     const GridDesc* __restrict__ grid,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals) {
  uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const GridDesc g = *grid;
  uint32_t cx = (uint32_t)cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
  uint32_t cy = (uint32_t)cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
  uint32_t cz = (uint32_t)cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
  keys[i] = morton3(cx, cy, cz);
  vals[i] = (uint32_t)i;
}

hipError_t morton_keys(const float* xyz, uint64_t n, const GridDesc* g0, uint32_t* keys,
                       uint32_t* vals, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_morton_keys, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz,
                     n, g0, keys, vals);
  return hipGetLastError();
}

// counts[cell of spts[j]] over the sorted points; consecutive points share a
// cell, so each wave adds one count per run of equal cells (one atomic per
// run instead of per point).
__global__ __launch_bounds__(256) void k_count_sorted(const float4* __restrict__ spts,
                                                      uint64_t n,
                                                      const GridDesc* __restrict__ grid,
                                                      uint32_t* __restrict__ counts) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  const GridDesc g = *grid;
  uint32_t key = 0xffffffffu;
  if (j < n) {
    const float4 p = spts[j];
    const int cx = cell_of(p.x, g.mn[0], g.inv, g.dim[0]);
    const int cy = cell_of(p.y, g.mn[1], g.inv, g.dim[1]);
    const int cz = cell_of(p.z, g.mn[2], g.inv, g.dim[2]);
    key = ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] + (uint32_t)cx;
  }
  const uint32_t prev = __shfl_up(key, 1, kWave);
  const bool head = j < n && (lane == 0 || prev != key);
  const uint64_t heads = __ballot(head);
  if (head) {
    // run ends at the next head (or at the end of the wave / of the data)
    const uint64_t after = lane == kWave - 1 ? 0ull : (heads >> (lane + 1)) << (lane + 1);
    const int next = after ? __ffsll((long long)after) - 1 : kWave;
    const uint64_t j0 = j - (uint64_t)lane;
    const uint64_t valid = min((uint64_t)kWave, n - j0);  // lanes holding points
    const uint32_t len = (uint32_t)(min((uint64_t)next, valid) - (uint64_t)lane);
    atomicAdd(&counts[key], len);
  }
}

hipError_t count_sorted(const float4* spts, uint64_t n, const GridDesc* g, uint32_t* counts,
                        hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_count_sorted, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, spts,
                     n, g, counts);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_count_cells(const float* __restrict__ xyz, uint64_t n,
                                                     const GridDesc* __restrict__ grid,
                                                     uint32_t* __restrict__ counts) {
  uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const GridDesc g = *grid;
  int cx = cell_of(xyz[3 * i], g.mn[0], g.inv, g.dim[0]);
  int cy = cell_of(xyz[3 * i + 1], g.mn[1], g.inv, g.dim[1]);
  int cz = cell_of(xyz[3 * i + 2], g.mn[2], g.inv, g.dim[2]);
  atomicAdd(&counts[((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] +
                    (uint32_t)cx],
            1u);
}

hipError_t count_cells(const float* xyz, uint64_t n, const GridDesc* g, uint32_t* counts,
                       hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_count_cells, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz,
                     n, g, counts);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_gather(const float* __restrict__ xyz,
                                                const uint32_t* __restrict__ vals, uint64_t n,
                                                float4* __restrict__ spts) {
  uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  uint32_t i = vals[j];
  spts[j] = make_float4(xyz[3ull * i], xyz[3ull * i + 1], xyz[3ull * i + 2],
                        __uint_as_float(i));
}

hipError_t gather_points(const float* xyz, const uint32_t* vals, uint64_t n, float4* spts,
                         hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, vals,
                     n, spts);
  return hipGetLastError();
}

// The grid by value, or (grid not null) planned on the device.
__global__ __launch_bounds__(256) void k_query_morton(const float* __restrict__ q, uint64_t nq,
                                                      const GridDesc gv,
                                                      const GridDesc* __restrict__ grid,
                                                      int shift, uint32_t* __restrict__ keys,
                                                      uint32_t* __restrict__ vals) {
  uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nq) return;
  const GridDesc g = grid ? *grid : gv;
  if (shift < 0) {
    // Grid planned on the device: 8 Morton bits per axis of the widest
    // axis's cell coordinate (the host's rule for a known grid).
    const uint32_t md = (uint32_t)max(max(g.dim[0], g.dim[1]), g.dim[2]) - 1u;
    const int bits = md ? 32 - __clz((int)md) : 0;
    shift = max(0, bits - 8);
  }
  // Queries outside the box (or NaN) clamp to the border cells.
  uint32_t cx = (uint32_t)cell_of(q[3 * i], g.mn[0], g.inv, g.dim[0]) >> shift;
  uint32_t cy = (uint32_t)cell_of(q[3 * i + 1], g.mn[1], g.inv, g.dim[1]) >> shift;
  uint32_t cz = (uint32_t)cell_of(q[3 * i + 2], g.mn[2], g.inv, g.dim[2]) >> shift;
  keys[i] = g.morton == 2 ? hilbert3(cx, cy, cz) : morton3(cx, cy, cz);
  vals[i] = (uint32_t)i;
}

hipError_t query_morton_keys(const float* q, uint64_t nq, const GridDesc& g, const GridDesc* gdev,
                             int shift, uint32_t* keys, uint32_t* vals, hipStream_t st) {
  if (nq == 0) return hipSuccess;
  hipLaunchKernelGGL(k_query_morton, dim3((uint32_t)((nq + 255) / 256)), dim3(256), 0, st, q,
                     nq, g, gdev, shift, keys, vals);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_morton(const uint32_t* __restrict__ xyz, uint64_t n,
                                                uint32_t* __restrict__ codes) {
  uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  codes[i] = morton3(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]);
}

hipError_t morton3_codes(const uint32_t* xyz, uint64_t n, uint32_t* codes, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_morton, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, xyz, n,
                     codes);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256)
    p[i] = v;
}

__global__ __launch_bounds__(256) void k_iota(uint32_t* __restrict__ p, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256)
    p[i] = (uint32_t)i;
}

static dim3 fill_grid(uint64_t n) {
  uint64_t b = (n + 255) / 256;
  return dim3((uint32_t)(b < 65536 ? (b ? b : 1) : 65536));
}

hipError_t fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, fill_grid(n), dim3(256), 0, st, p, n, v);
  return hipGetLastError();
}

hipError_t iota_u32(uint32_t* p, uint64_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_iota, fill_grid(n), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_scatter_rows(const float4* __restrict__ qproc,
                                                      const float* __restrict__ val, uint64_t n,
                                                      float r, float* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256)
    out[__float_as_uint(qproc[i].w)] = fminf(val[i], r);
}

hipError_t scatter_rows(const float4* qproc, const float* val, uint64_t n, float r, float* out,
                        hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_scatter_rows, fill_grid(n), dim3(256), 0, st, qproc, val, n, r, out);
  return hipGetLastError();
}

}  // namespace rtnn
