// Range search and KNN of up to 32 keys on a raster grid with the distance
// filter on the matrix cores (gfx950).
//
// A wave takes 64 consecutive queries, one per lane.  Queries next to each other
// share most of the points in their cells, so the wave loads the points of their
// cells' bounding block into LDS once and tests them against all 64: for 32
// points and 32 queries two v_mfma_f32_32x32x2 give R^2 - |q - p|^2 as
//   (x, y, z, -|p|^2) . (2x, 2y, 2z, 1) + (R^2 - |q|^2 + slack),
// coordinates taken from a query of the wave.  The slack exceeds every rounding
// of that sum, so its sign keeps all hits, and few points more.  One v_alignbit
// per element of the product collects the signs into masks, a v_permlane32_swap
// brings a query's two halves together, and a lane gets one word for 32 points, of
// which only the words with a bit set are kept.
//
// Each lane then takes its points one bit at a time, in batches of 16, computes
// d2 with d2_of's operations and tests it as every kernel here does.  The step of
// a batch is the register its key lives in, so no key passes through memory;
// batches are sorted and merged into the row in registers, all lanes at once
// (v_min_f64 / v_max_f64, see topk.h).
//
// A wave's latency bounds it at the 12 (K <= 16) or 8 waves per CU that its LDS
// and registers allow (learned KNN of 10M, K = 16: the matrix cores busy 0.14 of
// the time, VALU issue 0.56, a third of the wave cycles waiting for loads, LDS and
// stores).  Rows of 64 keys would need every register there
// is and spill (batches of 1024 clouds, K = 64: 20 ms against the group kernel's
// 13.6), so k > 32 stays with the groups.  A pass against groups of lanes per
// query, which test each query's candidates alone: 1M uniform points, r = 2.4,
// K = 32: 855 -> 437 us; 2M queries on sphere surfaces, K = 8: 1482 -> 686 us;
// learned KNN of 10M, K = 16: 5.23 -> 3.99 ms; 48 small clouds 167 -> 112 us.
#include <float.h>

#include <algorithm>

#include "common.h"
#include "internal.h"
#include "topk.h"

namespace rtnn {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kMatWaves = kTileQ / kWave;
constexpr int kMatTile = 32;   // points per product
// A wave's queries are taken together while their first cells lie within this
// many of the first one's: x is free along a row of cells (the block holds only
// the points there are), y and z multiply the rows.
constexpr int kSpanX = 16, kSpanYZ = 4;
constexpr int kBatch = 16;     // keys sorted at a time
constexpr int kStep = 8;       // of them read at a time

// Tiles listed before their hits are taken, and the waves per SIMD that their LDS
// and the row's registers leave.  K <= 16 has registers for three: 15 tiles make
// room for them (learned KNN of 10M 4.31 -> 3.99 ms against 24 and two).
template <int KC>
struct MatCfg {
  static constexpr int kTiles = KC <= 16 ? 15 : 24;
  static constexpr int kOccupancy = KC <= 16 ? 3 : 2;
};

// No key: what an empty slot of a row holds, d2 = inf and index -1.  Above every
// key, and as a double still finite.
__device__ inline double key_empty() { return key_double(__builtin_huge_valf(), ~0u); }

// a's upper 32 lanes exchanged with b's lower 32.
__device__ inline void swap_halves(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

// Writes the row's k keys.
template <int KC, bool KNN>
__device__ __forceinline__ void emit_row(const SearchArgs& a, const double (&list)[KC], bool active,
                                         uint32_t row, uint32_t qs, float R) {
  const uint32_t k = a.k;
  if (!active) return;
  int32_t* oi = a.out_idx + (uint64_t)row * k;
  float* od = a.out_d2 ? a.out_d2 + (uint64_t)row * k : nullptr;
  auto idx_of = [&](int i) { return (int)key_idx(key_bits(list[i])); };
  auto d2_at = [&](int i) { return key_d2(key_bits(list[i])); };
#pragma unroll
  for (int i = 0; i < KC; i += 4) {
    if ((uint32_t)i + 4u <= k) {
      *reinterpret_cast<i4u*>(oi + i) =
          i4u{idx_of(i), idx_of(i + 1), idx_of(i + 2), idx_of(i + 3)};
      if (od)
        *reinterpret_cast<f4u*>(od + i) = f4u{d2_at(i), d2_at(i + 1), d2_at(i + 2), d2_at(i + 3)};
    } else {
#pragma unroll
      for (int j = i; j < i + 3; ++j)
        if ((uint32_t)j < k) {
          oi[j] = idx_of(j);
          if (od) od[j] = d2_at(j);
        }
    }
  }
  if (KNN && a.short_rows) {  // (a range row is final)
    uint32_t hits = 0;
#pragma unroll
    for (int i = 0; i < KC; ++i)
      hits += (uint32_t)i < k && key_d2(key_bits(list[i])) < __builtin_huge_valf() ? 1u : 0u;
    append_short(a, hits < k && R < a.r, qs, hits, R);
  }
}

// The cells that a lane's query reaches (none: lo0 > hi0, or lo1 > hi1, ...).
struct CellBox {
  int lo0, hi0, lo1, hi1, lo2, hi2;
  __device__ bool some() const { return lo0 <= hi0 && lo1 <= hi1 && lo2 <= hi2; }
};
__device__ __forceinline__ CellBox cell_box(const GridDesc& g, const float4& q, float R) {
  CellBox c;
  cell_range(g, q.x, R, 0, c.lo0, c.hi0);
  cell_range(g, q.y, R, 1, c.lo1, c.hi1);
  cell_range(g, q.z, R, 2, c.lo2, c.hi2);
  return c;
}

// Block of the cells of a group of queries: those of `todo` near lane `lead`.
struct Block {
  uint32_t b0, b1, b2, e0, ny, rows;
};
__device__ __forceinline__ bool near_lead(const CellBox& c, int lead) {
  const int f0 = __builtin_amdgcn_readlane(c.lo0, lead);
  const int f1 = __builtin_amdgcn_readlane(c.lo1, lead);
  const int f2 = __builtin_amdgcn_readlane(c.lo2, lead);
  return abs(c.lo0 - f0) <= kSpanX && abs(c.lo1 - f1) <= kSpanYZ && abs(c.lo2 - f2) <= kSpanYZ;
}
__device__ __forceinline__ Block block_of(const CellBox& c, bool in) {
  Block b;
  b.b0 = wave_min_u32(in ? (uint32_t)c.lo0 : ~0u);
  b.b1 = wave_min_u32(in ? (uint32_t)c.lo1 : ~0u);
  b.b2 = wave_min_u32(in ? (uint32_t)c.lo2 : ~0u);
  b.e0 = wave_max_u32(in ? (uint32_t)c.hi0 : 0u);
  b.ny = wave_max_u32(in ? (uint32_t)c.hi1 : 0u) - b.b1 + 1u;
  b.rows = b.ny * (wave_max_u32(in ? (uint32_t)c.hi2 : 0u) - b.b2 + 1u);
  return b;
}
// Points s .. e of the block's row of cells j (none past the last row).
__device__ __forceinline__ void row_run(const SearchArgs& a, const GridDesc& g, const Block& b,
                                        uint32_t j, uint32_t& s, uint32_t& e) {
  s = 0;
  e = 0;
  if (j < b.rows) {
    const uint32_t rowc = g.cell_base + ((b.b2 + j / b.ny) * (uint32_t)g.dim[1] + b.b1 +
                                         j % b.ny) * (uint32_t)g.dim[0];
    s = a.cell_start[rowc + b.b0];
    e = a.cell_start[rowc + b.e0 + 1u];
  }
}

template <int KC, bool KNN>
__global__ __launch_bounds__(kTileQ)
__attribute__((amdgpu_waves_per_eu(MatCfg<KC>::kOccupancy))) void k_topk_matrix(
    const SearchArgs a) {
  constexpr int kTiles = MatCfg<KC>::kTiles;
  constexpr uint32_t kCap = kTiles * kMatTile;
  __shared__ float4 s_pts[kMatWaves][kCap];                  // listed points
  __shared__ uint32_t s_word[kMatWaves][kTiles + 1][kWave];  // a lane's non-zero words, then 0
  __shared__ uint8_t s_tile[kMatWaves][kTiles + 1][kWave];   // and their tiles
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int lane = threadIdx.x & (kWave - 1);
  const bool upper = lane >= kMatTile;
  float4* const pts = s_pts[w];
  // Product row i (lane i) takes point 16 (i / 4 % 2) + 4 (i / 8) + i % 4 of a
  // tile: element r of a lane's half h is then bit 16 h + r of the word.
  const uint32_t mine = (((uint32_t)lane >> 2) & 1u) * 16u + (((uint32_t)lane >> 3) & 3u) * 4u +
                        ((uint32_t)lane & 3u);
  const double none = key_empty();
  if (a.gate && *a.gate != 0) return;
  uint32_t q0, q1, gi;
  tile_of(a, a.nq, xcd_swizzle(blockIdx.x, gridDim.x), q0, q1, gi);
  const uint32_t qi = q0 + threadIdx.x;
  if (q0 + (uint32_t)w * kWave >= q1) return;
  const bool active = qi < q1;
  const uint32_t qs = active ? (a.qsel ? a.qsel[qi] : qi) : 0u;
  const GridDesc g = a.grids[gi];
  const float4 qv = active ? a.queries[qs] : make_float4(0.f, 0.f, 0.f, 0.f);
  const uint32_t row = __float_as_uint(qv.w);
  const float R = active ? query_radius(a, qi, qs) : a.r;
  const float R2 = R * R;
  float lim = r2_limit(R2);
  const CellBox cells = cell_box(g, qv, R);
  bool todo = active && cells.some();

  const uint32_t base = a.local_index ? g.point_base : 0u;
  double list[KC];
#pragma unroll
  for (int i = 0; i < KC; ++i) list[i] = none;

  uint32_t cnt = 0;     // points listed (whole tiles but the last)
  uint32_t tiles = 0;   // of them scanned
  uint32_t nw = 0;      // this lane's words
  // Takes the hits of the words, then starts over.
  auto collect = [&]() __attribute__((always_inline)) {
    s_word[w][nw][lane] = 0;
    uint32_t iw = 0, word = s_word[w][0][lane], tile = s_tile[w][0][lane];
    while (__ballot(word != 0) != 0) {
      // The next kBatch points of every lane.
      double v[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; b += kStep) {
        uint32_t c[kStep];
        float lm[kStep];
#pragma unroll
        for (int u = 0; u < kStep; ++u) {
          lm[u] = word != 0 ? lim : -1.0f;
          // a lane without a point left reads the first one listed (no hit)
          c[u] = word != 0 ? tile * kMatTile + (uint32_t)__builtin_ctz(word) : 0u;
          word &= word - 1u;  // 0 stays 0
          iw = min(iw + (word == 0 ? 1u : 0u), nw);
          const uint32_t next = s_word[w][iw][lane];
          tile = s_tile[w][iw][lane];
          word = word == 0 ? next : word;
        }
        float4 p[kStep];
#pragma unroll
        for (int u = 0; u < kStep; ++u) p[u] = pts[c[u]];
#pragma unroll
        for (int u = 0; u < kStep; ++u) {
          const float d2 = d2_of(qv.x, qv.y, qv.z, p[u].x, p[u].y, p[u].z);
          const bool hit = d2 <= lm[u] && (!KNN || d2 > 0.0f);
          v[b + u] = hit ? key_double(d2, __float_as_uint(p[u].w) - base) : none;
        }
      }
      sort_keys<kBatch>(v);
      merge_keys_inplace<KC, kBatch>(list, v);
      lim = fminf(lim, key_d2(key_bits(list[KC - 1])));
    }
    cnt = 0;
    tiles = 0;
    nw = 0;
    wave_sync();
  };

  // The group of queries at hand (in), the point its coordinates are taken
  // from, its side of the products, and what of its block is not listed yet:
  // rows of cells from rb on, the runs of the 64 rows before (one per lane,
  // `runs` those left) and points p0 .. p1 of one run.
  bool in = false, all = false;
  float cx = 0.f, cy = 0.f, cz = 0.f;
  float bx = 0.f, by = 0.f, bz = 0.f, one = 0.f, c0 = 0.f, c1 = 0.f;
  Block blk{0, 0, 0, 0, 1, 0};
  uint32_t rb = 0;
  uint32_t s = 0, e = 0, p0 = 0, p1 = 0;
  uint64_t runs = 0;
  bool last = false;
#pragma unroll 1
  while (!last) {
    if (rb >= blk.rows && runs == 0 && p0 == p1) {
      // The queries near the first one left, the block of their cells.
      const uint64_t left = __ballot(todo);
      if (left != 0) {
        const int lead = __builtin_ctzll(left);
        in = todo && near_lead(cells, lead);
        todo = todo && !in;
        blk = block_of(cells, in);
        rb = 0;
        cx = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(qv.x), lead));
        cy = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(qv.y), lead));
        cz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(qv.z), lead));
        // With M = |q|^2 + R^2 a hit has |p|^2 <= 2 M, no partial sum exceeds
        // 6 M, and all roundings together (of the sums, products, differences
        // from c, of R^2 and d2) stay below 80 * 2^-24 M; the slack is three
        // times that and covers underflow.  Where M is near overflow every
        // point is taken.
        bx = in ? qv.x - cx : 0.0f;
        by = in ? qv.y - cy : 0.0f;
        bz = in ? qv.z - cz : 0.0f;
        const float qq = fmaf(bx, bx, fmaf(by, by, bz * bz));
        const float M = qq + R2;
        all = __ballot(in && !(M < 0x1p+120f)) != 0;
        c0 = in ? (R2 - qq) + fmaf(M, 0x1p-16f, 0x1p-100f) : -FLT_MAX;
        c1 = c0;
        one = 1.0f;
        bx *= 2.0f;
        by *= 2.0f;
        bz *= 2.0f;
        swap_halves(bx, by);   // queries 0..31: bx, 32..63: by (x below, y above)
        swap_halves(bz, one);  // bz, one (z below, 1 above)
        swap_halves(c0, c1);
      } else {
        last = true;
      }
    }
    // List points until the list is full or the block is done.
    while (cnt < kCap) {
      if (p0 == p1) {
        if (runs == 0) {
          if (rb >= blk.rows) break;
          row_run(a, g, blk, rb + (uint32_t)lane, s, e);
          rb += kWave;
          runs = __ballot(e > s);
          continue;
        }
        const int rr = __builtin_ctzll(runs);
        runs &= runs - 1;
        p0 = (uint32_t)__builtin_amdgcn_readlane((int)s, rr);
        p1 = (uint32_t)__builtin_amdgcn_readlane((int)e, rr);
      }
      const uint32_t take = min(p1 - p0, kCap - cnt);
      // straight into LDS, 64 points a load, none waited for until the scan
      for (uint32_t j = 0; j < take; j += kWave)
        if (j + (uint32_t)lane < take)
          __builtin_amdgcn_global_load_lds(
              (const __attribute__((address_space(1))) void*)(a.spts + p0 + j + lane),
              (__attribute__((address_space(3))) void*)(pts + cnt + j), 16, 0, 0);
      cnt += take;
      p0 += take;
    }
    // (what the last tile holds past cnt gives no bit)
    const uint32_t full = (cnt + kMatTile - 1) / kMatTile * kMatTile;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    wave_sync();
    // The words of the tiles just listed.
    if (tiles * kMatTile < full) {
      f16v cv0, cv1;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        cv0[r] = c0;
        cv1[r] = c1;
      }
      // The next tile's points are on their way while one is multiplied.
      auto point = [&](uint32_t t) { return pts[min(t * kMatTile, full - kMatTile) + mine]; };
      float4 pa = point(tiles), pb;
      auto multiply = [&](const float4& p, float4& next) __attribute__((always_inline)) {
        const float x = p.x - cx, y = p.y - cy, z = p.z - cz;
        next = point(tiles + 1);
        const float n2 = fmaf(x, x, fmaf(y, y, z * z));
        const float a1 = upper ? y : x, a2 = upper ? -n2 : z;
        f16v d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, bx, cv0, 0, 0, 0);
        f16v d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, by, cv1, 0, 0, 0);
        d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2, bz, d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2, one, d1, 0, 0, 0);
        uint32_t m0 = 0, m1 = 0;
#pragma unroll
        for (int r = 15; r >= 0; --r)
          m0 = __builtin_amdgcn_alignbit(m0, __float_as_uint(d0[r]), 31);
#pragma unroll
        for (int r = 15; r >= 0; --r)
          m1 = __builtin_amdgcn_alignbit(m1, __float_as_uint(d1[r]), 31);
        const auto h = __builtin_amdgcn_permlane32_swap(m0, m1, false, false);
        const uint32_t miss = all ? 0u : h[0] | (h[1] << 16);
        const uint32_t have = cnt - tiles * kMatTile;  // of the tile's 32
        const uint32_t valid = have >= 32u ? ~0u : (1u << have) - 1u;
        const uint32_t word = in ? ~miss & valid : 0u;
        s_word[w][nw][lane] = word;
        s_tile[w][nw][lane] = (uint8_t)tiles;
        nw += word != 0 ? 1u : 0u;
        ++tiles;
      };
#pragma unroll 1
      for (;;) {
        multiply(pa, pb);
        if (tiles * kMatTile == full) break;
        multiply(pb, pa);
        if (tiles * kMatTile == full) break;
      }
      cnt = full;
    }
    if (last || cnt == kCap) collect();
  }

  emit_row<KC, KNN>(a, list, active, row, qs, R);
}

// Whether the queries suit this kernel, from up to 1024 waves spread over all:
// *use_groups becomes a.nq where groups of lanes are the better, 0 where it is
// (*told, which may be pinned host memory, 1 or 0).
//
// What decides is how many groups a wave's queries fall into, how many points
// these list and how many one query tests alone.  A wave of queries unlike the
// points (uniform ones over clumps, sparse ones on a fine grid) lists many for
// few tests, and the few waves that list the most are alone on the chip in the
// end.  The weights are fitted, in ns per wave, to 146 searches of 0.6 to 2
// million queries (uniform points, sphere surfaces, Gaussian clusters, Levy
// flights; queries as the points or uniform over their box).  The probe and the
// other kernel's empty launch take 12 us; with them the slowest choice takes 1.44
// times the faster kernel alone (queries mostly outside the points' box), the
// others at most 1.3 (searches of 50 us) and 1.15 from 200 us on.  By this kernel
// always, as by counts of points and queries alone, it was up to 9.5 times: 1M
// uniform queries over a Levy flight of 2M points, r = 2, K = 8, 469 us by groups,
// 4461 by this kernel, 487 with the probe.
constexpr int kProbeBlocks = 256, kProbeMaxGroups = 16;
constexpr int kProbeSums = 4;  // groups, listed points, their squares, own points
struct ProbeWeights {
  float group, listed, heaviest, base, own;
};

__global__ __launch_bounds__(kTileQ) void k_matrix_probe(const SearchArgs a, const ProbeWeights pw,
                                                         float* __restrict__ part,
                                                         uint32_t* __restrict__ ticket,
                                                         uint32_t* __restrict__ use_groups,
                                                         uint32_t* __restrict__ told) {
  __shared__ float s_v[kMatWaves][kProbeSums];
  __shared__ uint32_t s_last;
  const int w = (int)threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const uint32_t waves = (uint32_t)(((uint64_t)a.nq + kWave - 1) / kWave);
  const uint32_t probes = min(waves, (uint32_t)(kProbeBlocks * kMatWaves));
  const uint32_t me = blockIdx.x * kMatWaves + (uint32_t)w;
  float v[kProbeSums] = {};
  if (me < probes) {
    const uint32_t qi = (uint32_t)((uint64_t)me * waves / probes) * kWave + (uint32_t)lane;
    const bool active = qi < a.nq;
    const GridDesc g = a.grids[0];
    const float4 qv = active ? a.queries[qi] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float R = active ? query_radius(a, qi, qi) : a.r;
    const CellBox c = cell_box(g, qv, R);
    const bool some = active && c.some();
    bool todo = some;
    float listed = 0.0f, own = 0.0f;
    int groups = 0;
    for (uint64_t left = __ballot(todo); left != 0 && groups < kProbeMaxGroups;
         left = __ballot(todo), ++groups) {
      const bool in = todo && near_lead(c, __builtin_ctzll(left));
      todo = todo && !in;
      const Block b = block_of(c, in);
      for (uint32_t j = (uint32_t)lane; j < b.rows; j += kWave) {
        uint32_t s, e;
        row_run(a, g, b, j, s, e);
        listed += (float)(e - s);
      }
    }
    // eight of the queries alone, 16 lanes each
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int src = (lane & ~15) + 8 * h + 4;
      const int w0 = __shfl(c.lo0, src, kWave), w1 = __shfl(c.lo1, src, kWave),
                w2 = __shfl(c.lo2, src, kWave), x0 = __shfl(c.hi0, src, kWave),
                x1 = __shfl(c.hi1, src, kWave), x2 = __shfl(c.hi2, src, kWave);
      const int sy = x1 - w1 + 1;
      const int rows = __shfl(some ? 1 : 0, src, kWave) * sy * (x2 - w2 + 1);
      for (int j = lane & 15; j < rows; j += 16) {
        const uint32_t rowc = g.cell_base + ((uint32_t)(w2 + j / sy) * (uint32_t)g.dim[1] +
                                             (uint32_t)(w1 + j % sy)) * (uint32_t)g.dim[0];
        own += (float)(a.cell_start[rowc + x0 + 1] - a.cell_start[rowc + w0]);
      }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
      listed += __shfl_xor(listed, o, kWave);
      own += __shfl_xor(own, o, kWave);
    }
    v[0] = (float)groups;
    v[1] = listed;
    v[2] = listed * listed;
    v[3] = own * 0.125f;
  }
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < kProbeSums; ++i) s_v[w][i] = v[i];
  __syncthreads();
  // Folded by the last block to finish, as in k_bbox.
  if (threadIdx.x == 0) {
    for (int i = 0; i < kProbeSums; ++i) {
      float t = 0.0f;
      for (int u = 0; u < kMatWaves; ++u) t += s_v[u][i];
      __hip_atomic_store(&part[kProbeSums * blockIdx.x + i], t, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             gridDim.x - 1;
  }
  __syncthreads();
  if (!s_last || w != 0) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
  for (int i = 0; i < kProbeSums; ++i) v[i] = 0.0f;
  for (uint32_t b = (uint32_t)lane; b < gridDim.x; b += kWave)
#pragma unroll
    for (int i = 0; i < kProbeSums; ++i)
      v[i] += __hip_atomic_load(&part[kProbeSums * b + i], __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1)
#pragma unroll
    for (int i = 0; i < kProbeSums; ++i) v[i] += __shfl_xor(v[i], o, kWave);
  if (lane == 0) {
    const float each = 1.0f / (float)probes;
    const float here = pw.group * v[0] * each + pw.listed * v[1] * each +
                       pw.heaviest * v[2] / (fmaxf(v[1], 1.0f) * (float)waves);
    const bool groups = here > pw.base + pw.own * v[3] * each;
    *use_groups = groups ? a.nq : 0u;
    *told = groups ? 1u : 0u;
    __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

hipError_t matrix_probe(const SearchArgs& a, bool knn, float* part, uint32_t* ticket,
                        uint32_t* use_groups, uint32_t* told, hipStream_t st) {
  if (a.tiles || a.nq == 0) return hipErrorInvalidValue;
  static_assert(kProbeBlocks * kProbeSums * 4 <= kBboxPartBytes, "partial sums");
  const ProbeWeights pw = knn ? ProbeWeights{0.2f, 0.0128f, 3.0f, 4.5f, 0.094f}
                              : ProbeWeights{2.5f, 0.006f, 30.0f, 12.0f, 0.05f};
  hipLaunchKernelGGL(k_matrix_probe, dim3(kProbeBlocks), dim3(kTileQ), 0, st, a, pw, part, ticket,
                     use_groups, told);
  return hipGetLastError();
}

template <int KC>
static void launch_matrix_kc(const SearchArgs& a, bool knn, dim3 grid, hipStream_t st) {
  if (knn)
    hipLaunchKernelGGL((k_topk_matrix<KC, true>), grid, dim3(kTileQ), 0, st, a);
  else
    hipLaunchKernelGGL((k_topk_matrix<KC, false>), grid, dim3(kTileQ), 0, st, a);
}

hipError_t launch_matrix(const SearchArgs& a0, bool knn, hipStream_t st) {
  SearchArgs a = a0;
  if (a.k == 0 || a.k > 32 || a.nlevels > 0 || a.nq_dev) return hipErrorInvalidValue;
  if (!a.tiles) {
    a.tile_q = (uint32_t)kTileQ;
    a.ntiles = (uint32_t)(((uint64_t)a.nq + kTileQ - 1) / kTileQ);
  }
  if (a.ntiles == 0) return hipSuccess;
  const dim3 grid(a.ntiles);
  if (a.k <= 16) launch_matrix_kc<16>(a, knn, grid, st);
  else launch_matrix_kc<32>(a, knn, grid, st);
  return hipGetLastError();
}

}  // namespace rtnn
