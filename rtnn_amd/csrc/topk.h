// Device helpers of the top-k kernels: query tiles, wave reductions, keys as
// doubles, query radius, the short-row list.
#pragma once

#include "common.h"

namespace rtnn {

__device__ inline uint64_t lanemask_lt64() {
  const int lane = threadIdx.x & (kWave - 1);
  return lane == 0 ? 0ull : (~0ull >> (kWave - lane));
}

// d2 < R2 as d2 <= r2_limit(R2): the float just below R2 (-1 for R2 <= 0,
// FLT_MAX for +inf).  After a select the limit becomes the k-th key's d2:
// ties with it are appended too and resolved by the (d2, index) rank.
__device__ inline float r2_limit(float R2) {
  return R2 > 0.0f ? __uint_as_float(__float_as_uint(R2) - 1u) : -1.0f;
}

// Query count of this launch (device-resident for the fallback pass).
__device__ inline uint32_t launch_nq(const SearchArgs& a) {
  return a.nq_dev ? *a.nq_dev : a.nq;
}

// Appends the processing positions of short rows (fewer than k hits) with
// one atomic per wave; a wave's entries stay together and in lane order, so
// the re-run over the list keeps the Morton locality of the queries.
__device__ inline void append_short(const SearchArgs& a, bool is_short, uint32_t qs,
                                    uint32_t hits, float R) {
  const uint64_t m = __ballot(is_short);
  if (m == 0) return;
  const int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0;
  if ((int)(threadIdx.x & (kWave - 1)) == leader)
    base = atomicAdd(a.short_count, (uint32_t)__popcll(m));
  base = __shfl(base, leader, kWave);
  if (is_short) {
    const uint32_t pos = base + (uint32_t)__popcll(m & lanemask_lt64());
    a.short_rows[pos] = qs;
    if (a.short_hits) a.short_hits[pos] = hits;
    if (a.radius_out) a.radius_out[qs] = R;
  }
}

// Search radius of launch position qi (query qs).
__device__ inline float query_radius(const SearchArgs& a, uint32_t qi, uint32_t qs) {
  if (!a.qradius) return a.r;
  const float sc = a.qsel_hits ? hit_scale(a.qsel_hits[qi], a.k) : a.qradius_scale;
  return fminf(a.r, a.qradius[qs] * sc);
}

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Resolves tile t into its query range and grid.
__device__ __forceinline__ void tile_of(const SearchArgs& a, uint32_t nq, uint32_t t, uint32_t& q0,
                               uint32_t& q1, uint32_t& gi) {
  if (a.tiles) {
    Tile tl = a.tiles[t];
    q0 = tl.q0; q1 = tl.q1; gi = tl.grid;
  } else {
    q0 = t * a.tile_q;
    q1 = min(q0 + a.tile_q, nq);
    gi = 0;
  }
}

// Persistent launches walk tiles in XCD-contiguous chunks; plain launches map
// each block to one tile through xcd_swizzle.
struct TileIter {
  uint32_t t, end, step;
  __device__ __forceinline__ TileIter(const SearchArgs& a, uint32_t nq) {
    uint32_t ntiles = a.nq_dev ? (nq + a.tile_q - 1) / a.tile_q : a.ntiles;
    if (a.persistent) {
      constexpr uint32_t kXcd = 8;
      uint32_t x = blockIdx.x % kXcd, j = blockIdx.x / kXcd;
      uint32_t per = (gridDim.x + kXcd - 1 - x) / kXcd;  // blocks on this XCD
      uint32_t q = ntiles / kXcd, rem = ntiles % kXcd;
      uint32_t start = x * q + (x < rem ? x : rem);
      end = start + q + (x < rem ? 1u : 0u);
      t = start + j;
      step = per;
    } else {
      t = xcd_swizzle(blockIdx.x, gridDim.x);
      end = t + 1;
      step = 1;
    }
  }
};

// ---- wave reductions

// Lane moves that leave the identity of an unsigned minimum where no lane is
// read, so that each folds into its v_min_u32.
template <int CTRL, int ROWS>
__device__ inline uint32_t dpp_or_max(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, ROWS, 0xf, false);
}
// Minimum over the wave, uniform (row shifts, then the two row broadcasts).
__device__ inline uint32_t wave_min_u32(uint32_t v) {
  v = min(v, dpp_or_max<0x111, 0xf>(v));
  v = min(v, dpp_or_max<0x112, 0xf>(v));
  v = min(v, dpp_or_max<0x114, 0xf>(v));
  v = min(v, dpp_or_max<0x118, 0xf>(v));
  v = min(v, dpp_or_max<0x142, 0xa>(v));
  v = min(v, dpp_or_max<0x143, 0xc>(v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
__device__ inline uint32_t wave_max_u32(uint32_t v) { return ~wave_min_u32(~v); }

// ---- keys as doubles
//
// A key (d2 bits << 32 | index) of a finite d2 >= 0 is the bit pattern of a
// non-negative finite double (its exponent field is at most 0x7f7), and
// non-negative doubles order like their bits, denormals included.  Minimum
// and maximum are then one full-rate instruction each where a 64-bit integer
// compare-exchange takes a compare and four selects.  The instructions are
// named in asm because fmin / fmax would first quiet every operand.
__device__ inline double key_double(float d2, uint32_t idx) {
  return __longlong_as_double((long long)pack_key(d2, idx));
}
__device__ inline uint64_t key_bits(double k) { return (uint64_t)__double_as_longlong(k); }
// No key: +infinity, above every key.
__device__ inline double key_none() { return __builtin_huge_val(); }

__device__ inline double key_min(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// a, b <- the smaller, the larger.
__device__ inline void key_cx(double& a, double& b) {
  double lo;
  asm volatile("v_min_f64 %0, %2, %1\n\tv_max_f64 %1, %2, %1" : "=&v"(lo), "+v"(b) : "v"(a));
  a = lo;
}

// The same with a and b in the registers they are in, for a list that lives
// across a loop: with key_cx its keys change registers, and the copies back at
// the loop's joins were spilled.
__device__ inline void key_cx_inplace(double& a, double& b) {
  double lo;
  asm volatile("v_min_f64 %0, %1, %2\n\tv_max_f64 %2, %1, %2\n\tv_mov_b64 %1, %0"
               : "=&v"(lo), "+v"(a), "+v"(b));
}

// Sorts N keys ascending: Batcher's odd-even merge sort of the next power of
// two, whose missing last keys would be the largest (12 keys: 42
// compare-exchanges).  One comparator level per template instance,
// so that every index is a constant and the keys stay in registers.
template <int N, int P, int Q>
__device__ __forceinline__ void sort_level(double (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N - Q; ++i) {
    const int off = i - Q % P;
    if (off >= 0 && off % (2 * Q) < Q && i / (2 * P) == (i + Q) / (2 * P)) key_cx(v[i], v[i + Q]);
  }
  if constexpr (Q > 1)
    sort_level<N, P, Q / 2>(v);
  else if constexpr (2 * P < N)
    sort_level<N, 2 * P, 2 * P>(v);
}
template <int N>
__device__ __forceinline__ void sort_keys(double (&v)[N]) {
  sort_level<N, 1, 1>(v);
}

template <int KC, int H>
__device__ __forceinline__ void bitonic_level(double (&list)[KC]) {
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if ((i & H) == 0) key_cx(list[i], list[i + H]);
  if constexpr (H > 1) bitonic_level<KC, H / 2>(list);
}

// list <- the KC smallest of list and v, both ascending: each of the list's
// last keys against v reversed leaves a bitonic sequence of the smallest,
// which a bitonic merge orders.
template <int KC, int NB>
__device__ __forceinline__ void merge_keys(double (&list)[KC], const double (&v)[NB]) {
#pragma unroll
  for (int i = 0; i < (KC < NB ? KC : NB); ++i)
    list[KC - 1 - i] = key_min(list[KC - 1 - i], v[i]);
  bitonic_level<KC, KC / 2>(list);
}

// The same on a list that keeps its registers.
template <int KC, int H>
__device__ __forceinline__ void bitonic_level_inplace(double (&list)[KC]) {
#pragma unroll
  for (int i = 0; i < KC; ++i)
    if ((i & H) == 0) key_cx_inplace(list[i], list[i + H]);
  if constexpr (H > 1) bitonic_level_inplace<KC, H / 2>(list);
}
template <int KC, int NB>
__device__ __forceinline__ void merge_keys_inplace(double (&list)[KC], const double (&v)[NB]) {
#pragma unroll
  for (int i = 0; i < (KC < NB ? KC : NB); ++i)
    asm volatile("v_min_f64 %0, %0, %1" : "+v"(list[KC - 1 - i]) : "v"(v[i]));
  bitonic_level_inplace<KC, KC / 2>(list);
}

}  // namespace rtnn
