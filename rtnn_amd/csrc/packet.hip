// KNN by packets of 64 queries over a tree of bounding boxes (gfx950).
//
// The points are sorted along a Hilbert curve, so every run of consecutive
// points is compact: kLeafPts of them form a leaf with its box, kFan leaves a
// level-1 node, kFan of those a level-2 node and so on.  Nothing depends on the
// radius or on a cell size, and no per-cell table is built.  (Morton order,
// whose runs jump, needs 1.6 times the leaves: 72 against 46 of 16 points per
// packet on a Gaussian mixture at K = 8.)
//
// A wave takes 64 queries that are neighbours on the curve, one per lane, and
// walks the tree once for all of them: the path is wave-uniform, so no lane
// waits for another's loop.  At a node lane c tests child c's box against the
// box of the packet, then each child in reach is tested against every lane's
// query and limit, its box in scalars.  The walk needs good limits, so every
// lane first scans the leaves around the one nearest to it.
//
// Hits go to a small LDS column per lane and are merged into the lane's sorted
// list in batches, all lanes at once.  Keys (d2 bits << 32 | index) are
// positive doubles whose order is the keys' order, so a compare-exchange is
// v_min_f64 and v_max_f64, both full rate on this chip: a merge of up to
// 16 keys into 16 costs about 210 instructions per wave where inserting keys
// one by one cost about 100 per key with most lanes idle.
//
// VALU issue bounds it (0.9 of its cycles on sphere surfaces, K = 16).  Against
// one query per lane over the cells of a grid of edge r (a pass, 1M points and
// queries): Gaussian mixture r = 20, K = 8: 10.5 -> 0.92 ms, K = 50: 153 ->
// 3.5; sphere surfaces r = 10, K = 16 (4M): 4.73 -> 2.14; uniform points with
// fewer hits than K in r are the one case where the cells are as fast.
//
// Exactness: a box distance is computed by the operations of d2_of on the
// nearest corner, and every one of them is monotone in FP32, so it never
// exceeds the d2 of a point inside; a box is skipped only beyond the limit.
#include <algorithm>

#include "common.h"
#include "internal.h"
#include "topk.h"

namespace rtnn {

// ------------------------------------------------------------------ build

// Boxes of one block's kFan leaves (kFan * kLeafPts consecutive points) and of
// their level-1 node, over the points it gathers into sorted order.  Positions
// past n get points at infinity (never a hit; a leaf is read whole), and
// leaves past the last an empty box that no limit reaches.
constexpr int kNodePts = kFan * kLeafPts;

__device__ inline void box_reduce(float (&mn)[3], float (&mx)[3], int width) {
  for (int o = width / 2; o > 0; o >>= 1) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      mn[a] = fminf(mn[a], __shfl_xor(mn[a], o, kWave));
      mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], o, kWave));
    }
  }
}

__global__ __launch_bounds__(256) void k_gather_boxes(const float* __restrict__ xyz,
                                                      const uint32_t* __restrict__ vals,
                                                      uint64_t n, float4* __restrict__ spts,
                                                      float4* __restrict__ box0,
                                                      float4* __restrict__ box1) {
  __shared__ float s_mn[256 / kWave][3], s_mx[256 / kWave][3];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const uint64_t base = (uint64_t)blockIdx.x * kNodePts;
  const float inf = __builtin_huge_valf();
  float nmn[3] = {inf, inf, inf}, nmx[3] = {-inf, -inf, -inf};
  static_assert(kNodePts % 256 == 0 && kWave % kLeafPts == 0, "whole leaves per wave");
#pragma unroll
  for (int u = 0; u < kNodePts / 256; ++u) {
    const uint64_t j = base + (uint64_t)(u * 256) + threadIdx.x;
    float mn[3] = {inf, inf, inf}, mx[3] = {-inf, -inf, -inf};
    float4 p = make_float4(inf, inf, inf, __uint_as_float(0xffffffffu));
    if (j < n) {
      const uint32_t i = vals[j];
      p = make_float4(xyz[3ull * i], xyz[3ull * i + 1], xyz[3ull * i + 2], __uint_as_float(i));
      mn[0] = mx[0] = p.x;
      mn[1] = mx[1] = p.y;
      mn[2] = mx[2] = p.z;
    }
    const uint64_t leaf = j / kLeafPts;
    const uint64_t nleaf = (n + kLeafPts - 1) / kLeafPts;
    if (leaf < nleaf) spts[j] = p;
    box_reduce(mn, mx, kLeafPts);
    if (leaf < nleaf && lane % kLeafPts == 0) {
      box0[2 * leaf] = make_float4(mn[0], mn[1], mn[2], 0.0f);
      box0[2 * leaf + 1] = make_float4(mx[0], mx[1], mx[2], 0.0f);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      nmn[a] = fminf(nmn[a], mn[a]);
      nmx[a] = fmaxf(nmx[a], mx[a]);
    }
  }
  box_reduce(nmn, nmx, kWave);
  if (lane == 0)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      s_mn[w][a] = nmn[a];
      s_mx[w][a] = nmx[a];
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 256 / kWave; ++i)
      for (int a = 0; a < 3; ++a) {
        s_mn[0][a] = fminf(s_mn[0][a], s_mn[i][a]);
        s_mx[0][a] = fmaxf(s_mx[0][a], s_mx[i][a]);
      }
    box1[2 * blockIdx.x] = make_float4(s_mn[0][0], s_mn[0][1], s_mn[0][2], 0.0f);
    box1[2 * blockIdx.x + 1] = make_float4(s_mx[0][0], s_mx[0][1], s_mx[0][2], 0.0f);
  }
}

// One wave per node: the box of its (up to) kFan children.
__global__ __launch_bounds__(256) void k_node_boxes(const float4* __restrict__ child,
                                                    uint32_t nchild, uint32_t nnode,
                                                    float4* __restrict__ box) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t node = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  if (node >= nnode) return;
  const uint32_t c = node * kFan + (uint32_t)lane;
  const float inf = __builtin_huge_valf();
  float mn[3] = {inf, inf, inf}, mx[3] = {-inf, -inf, -inf};
  if (c < nchild) {
    const float4 lo = child[2ull * c], hi = child[2ull * c + 1];
    mn[0] = lo.x; mn[1] = lo.y; mn[2] = lo.z;
    mx[0] = hi.x; mx[1] = hi.y; mx[2] = hi.z;
  }
  box_reduce(mn, mx, kWave);
  if (lane == 0) {
    box[2ull * node] = make_float4(mn[0], mn[1], mn[2], 0.0f);
    box[2ull * node + 1] = make_float4(mx[0], mx[1], mx[2], 0.0f);
  }
}

BoxTree box_tree_layout(uint64_t n, float4* box) {
  BoxTree t{};
  t.box = box;
  uint64_t c = (n + kLeafPts - 1) / kLeafPts, off = 0;
  for (int l = 0; l < kTreeLevels; ++l) {
    t.off[l] = (uint32_t)off;
    t.cnt[l] = (uint32_t)c;
    t.top = l;
    off += c;
    if (l >= 1 && c <= (uint64_t)kFan) break;  // level 1 is always built
    c = (c + kFan - 1) / kFan;
  }
  t.boxes = off;
  return t;
}

hipError_t build_box_tree(const float* xyz, const uint32_t* vals, uint64_t n, float4* spts,
                          const BoxTree& t, hipStream_t st) {
  if (n == 0) return hipSuccess;
  float4* box = const_cast<float4*>(t.box);
  hipLaunchKernelGGL(k_gather_boxes, dim3(t.cnt[1]), dim3(256), 0, st, xyz, vals, n, spts,
                     box + 2ull * t.off[0], box + 2ull * t.off[1]);
  for (int l = 2; l <= t.top; ++l)
    hipLaunchKernelGGL(k_node_boxes, dim3((t.cnt[l] + 3) / 4), dim3(256), 0, st,
                       box + 2ull * t.off[l - 1], t.cnt[l - 1], t.cnt[l], box + 2ull * t.off[l]);
  return hipGetLastError();
}

// ------------------------------------------------------------------- walk

// Read-only data at a wave-uniform address, through scalar loads.
typedef float f4v __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) f4v* const_f4;
__device__ inline const_f4 uniform_ptr(const float4* p, uint32_t i) {
  return (const_f4)(p + (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)i));
}

__device__ inline float wave_min_f(float v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, kWave));
  return v;
}
__device__ inline float wave_max_f(float v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}

// d2_of's operations on the distance to a box.
__device__ inline float gap_d2(float gx, float gy, float gz) {
  const float sx = gx * gx, sy = gy * gy, sz = gz * gz;
  const float s = sx + sy;
  return s + sz;
}

constexpr int kPacketWaves = 4;
constexpr int kLeafStep = 4;  // points tested between two looks at the buffers

// How the chosen leaves are tested.  kOwn: each lane queues the leaves within
// its own limit and the lanes scan one leaf each, by gathers; else every lane
// tests every leaf that some lane needs, from scalar loads.  A leaf is needed
// by 12 of 64 lanes on average, so scanning apart does a quarter of the tests,
// but each of its loads takes the vector data path 64 ways: it pays where few
// keys are kept.  1M uniform points and queries: K = 4 0.22 against 0.32 ms,
// K = 8 0.25 / 0.33 (0.28 / 0.31 on sphere surfaces); 4M on sphere surfaces,
// K = 16: 2.54 / 1.67 ms.
template <int KC>
struct PacketCfg {
  static constexpr bool kOwn = KC <= 8;
  static constexpr int kBuf = kOwn ? 12 : 16;  // keys per lane between merges
  static constexpr int kQueue = kOwn ? 8 : 1;  // leaves waiting per lane
  // Waves per SIMD: what 40 KB of LDS per block and a list of 2 KC registers
  // leave (K = 16: 128 VGPRs, 88 bytes of scratch, 2.19 ms a pass at 4M on sphere
  // surfaces against 2.39 at three waves).
  static constexpr int kOccupancy = KC <= 16 ? 4 : KC <= 32 ? 2 : 1;
};

template <int KC>
__global__ __launch_bounds__(kPacketWaves * kWave)
__attribute__((amdgpu_waves_per_eu(PacketCfg<KC>::kOccupancy))) void k_knn_packet(
    const SearchArgs a, const BoxTree t) {
  using C = PacketCfg<KC>;
  // Row i of a wave's buffer holds key i of every lane (a lane's column is its
  // own two banks at every row).  The last row only takes the write past the
  // last hit.
  __shared__ double s_buf[kPacketWaves][C::kBuf][kWave];
  __shared__ uint32_t s_que[kPacketWaves][C::kQueue][C::kOwn ? kWave : 1];  // a ring per lane
  __shared__ uint2 s_key[kPacketWaves][kTreeLevels - 2][kWave];  // levels 2 and up
  const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const uint32_t k = a.k;
  const uint32_t nq = launch_nq(a);
  const uint32_t nblk = gridDim.x;
  // Queries per wave: 64 where there are enough of them, else as many as spread
  // them over all waves of the grid.  Few queries (and the short rows of a list) are
  // far apart: the fewer a wave takes, the less of the tree it walks for queries
  // that it has not, and the more CUs walk (1000 queries over 300k uniform points,
  // K = 8: 905 us by packets of 64, 210 one per wave; 10,000 points as queries, K =
  // 64: 204 / 159).
  const uint32_t per =
      min((nq + nblk * kPacketWaves - 1) / (nblk * kPacketWaves), (uint32_t)kWave);
  const uint32_t ntiles = per ? (nq + per - 1) / per : 0u;
  char* const col = reinterpret_cast<char*>(&s_buf[w][0][lane]);
  auto at = [&](uint32_t o) -> double& { return *reinterpret_cast<double*>(col + o); };
  constexpr uint32_t kRow = 8 * kWave;  // bytes between a column's keys
  const double none = key_none();
#pragma unroll
  for (int i = 0; i < C::kBuf; ++i) at(i * kRow) = none;

  // Wave tiles: one per wave, or grid-strided where the count is on the device.
  for (uint32_t tb = xcd_swizzle(blockIdx.x, nblk);; tb += nblk) {
    const uint32_t tile = tb * kPacketWaves + (uint32_t)w;
    if (tile >= ntiles) break;
    const uint32_t qi = tile * per + (uint32_t)lane;
    const bool active = qi < nq && (uint32_t)lane < per;
    const uint32_t qs = active ? (a.qsel ? a.qsel[qi] : qi) : 0u;
    const float4 qv = active ? a.queries[qs] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t row = __float_as_uint(qv.w);
    const float R = active ? query_radius(a, qi, qs) : a.r;
    // A query at infinity or NaN has no hit: it takes no part in the walk.
    const bool live = active && isfinite(qv.x) && isfinite(qv.y) && isfinite(qv.z);
    float lim = live ? r2_limit(R * R) : -1.0f;
    const float inf = __builtin_huge_valf();
    const float plx = wave_min_f(live ? qv.x : inf), phx = wave_max_f(live ? qv.x : -inf);
    const float ply = wave_min_f(live ? qv.y : inf), phy = wave_max_f(live ? qv.y : -inf);
    const float plz = wave_min_f(live ? qv.z : inf), phz = wave_max_f(live ? qv.z : -inf);
    // list[KC - k ..] are the k smallest keys so far; the slots before them
    // hold zero (below every key), so list[KC - 1] is the k-th.
    double list[KC];
#pragma unroll
    for (int i = 0; i < KC; ++i) list[i] = (uint32_t)i < (uint32_t)KC - k ? 0.0 : none;
    uint32_t slot = 0;  // byte offset of the next free key of the column
    // limits are >= 0 or -1 (no hit): compared as unsigned with -1 -> 0
    uint32_t maxlim = wave_max_u32(lim < 0.0f ? 0u : __float_as_uint(lim));

    auto merge = [&]() __attribute__((always_inline)) {
      at(slot) = none;
      double v[C::kBuf];
#pragma unroll
      for (int i = 0; i < C::kBuf; ++i) v[i] = at(i * kRow);
      sort_keys<C::kBuf>(v);
      merge_keys<KC, C::kBuf>(list, v);
#pragma unroll
      for (int i = 0; i < C::kBuf; ++i) at(i * kRow) = none;
      slot = 0;
      const uint64_t last = key_bits(list[KC - 1]);
      if (last < key_bits(none)) lim = fminf(lim, key_d2(last));
    };
    auto room = [&]() __attribute__((always_inline)) {
      if (__ballot(slot >= (uint32_t)(C::kBuf - kLeafStep) * kRow) != 0) merge();
    };
    // One point against the lane's limit: every lane writes its key to its next
    // free place and moves on only past a hit (no branch).
    auto test = [&](float x, float y, float z, float idx, float lm) {
      const float d2 = d2_of(qv.x, qv.y, qv.z, x, y, z);
      at(slot) = key_double(d2, __float_as_uint(idx));
      slot += (d2 > 0.0f && d2 <= lm) ? kRow : 0u;
    };
    // The points of one leaf per lane (each its own), all lanes together; a
    // lane that has none passes any leaf and on = false.
    auto scan = [&](uint32_t leaf, bool on) __attribute__((always_inline)) {
      const float4* p = a.spts + (uint64_t)leaf * kLeafPts;
#pragma unroll 1
      for (int g = 0; g < kLeafPts; g += kLeafStep, p += kLeafStep) {
        float4 pv[kLeafStep];
#pragma unroll
        for (int u = 0; u < kLeafStep; ++u) pv[u] = p[u];
        room();
        const float lm = on ? lim : -1.0f;
#pragma unroll
        for (int u = 0; u < kLeafStep; ++u) test(pv[u].x, pv[u].y, pv[u].z, pv[u].w, lm);
      }
    };

    if (__ballot(lim >= 0.0f) != 0) {
      const float pmx = 0.5f * plx + 0.5f * phx, pmy = 0.5f * ply + 0.5f * phy,
                  pmz = 0.5f * plz + 0.5f * phz;
      // This lane's child of the node at hand: squared distance from the
      // packet's middle (bits | lane; the visiting order) and from the packet's
      // box (the bound), ~0 when it is done.
      uint32_t ckey = ~0u, cgap = ~0u;
      auto gap_of = [&](const float4& blo, const float4& bhi) {
        const float gx = fmaxf(fmaxf(blo.x - phx, plx - bhi.x), 0.0f);
        const float gy = fmaxf(fmaxf(blo.y - phy, ply - bhi.y), 0.0f);
        const float gz = fmaxf(fmaxf(blo.z - phz, plz - bhi.z), 0.0f);
        return __float_as_uint(gap_d2(gx, gy, gz));
      };
      auto mid_of = [&](const float4& blo, const float4& bhi) {
        const float cx = fmaxf(fmaxf(blo.x - pmx, pmx - bhi.x), 0.0f);
        const float cy = fmaxf(fmaxf(blo.y - pmy, pmy - bhi.y), 0.0f);
        const float cz = fmaxf(fmaxf(blo.z - pmz, pmz - bhi.z), 0.0f);
        return (__float_as_uint(gap_d2(cx, cy, cz)) & ~(uint32_t)(kFan - 1)) | (uint32_t)lane;
      };
      // Distance of this lane's query from a box given in scalars.
      auto lane_gap = [&](float lx, float ly, float lz, float hx, float hy, float hz) {
        const float gx = fmaxf(fmaxf(lx - qv.x, qv.x - hx), 0.0f);
        const float gy = fmaxf(fmaxf(ly - qv.y, qv.y - hy), 0.0f);
        const float gz = fmaxf(fmaxf(lz - qv.z, qv.z - hz), 0.0f);
        return gap_d2(gx, gy, gz);
      };
      auto expand = [&](int lvl, uint32_t node) {
        const uint32_t c = node * kFan + (uint32_t)lane;
        cgap = ~0u;
        if (c < t.cnt[lvl]) {
          const float4* b = t.box + 2ull * (t.off[lvl] + c);
          const float4 blo = b[0], bhi = b[1];
          cgap = gap_of(blo, bhi);
          ckey = mid_of(blo, bhi);
        }
      };
      // Children of `node` at level lvl in the order of mid_of, down to the
      // level-1 nodes; leaves(child) handles one of those and says whether to
      // go on.  reach() is the bound on the gap.
      auto walk = [&](auto&& reach, auto&& leaves) {
        int lvl = t.top;    // level of the children being visited
        uint32_t node = 0;  // their parent (index among level lvl + 1)
        expand(lvl, node);
        for (;;) {
          const uint32_t m = wave_min_u32(cgap <= reach() ? ckey : ~0u);
          if (m == ~0u) {  // none left within reach
            if (lvl == t.top) break;
            ++lvl;
            ckey = s_key[w][lvl - 2][lane].x;
            cgap = s_key[w][lvl - 2][lane].y;
            node = node / kFan;  // the parent of the node just left
            continue;
          }
          const uint32_t cl = m & (uint32_t)(kFan - 1);
          if ((uint32_t)lane == cl) cgap = ~0u;
          const uint32_t child = node * kFan + cl;
          // near some lane?
          const_f4 cb = uniform_ptr(t.box, 2u * (t.off[lvl] + child));
          const f4v lo = cb[0], hi = cb[1];
          if (__ballot(lane_gap(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z) <= lim) == 0) continue;
          if (lvl > 1) {
            s_key[w][lvl - 2][lane] = make_uint2(ckey, cgap);
            --lvl;
            node = child;
            expand(lvl, node);
          } else if (!leaves(child)) {
            break;
          }
        }
      };
      // The leaves of level-1 node `child` whose gap from the packet's box is at
      // most `reach`, one after the other: f(leaf, distance of this lane's query
      // from its box).  Lane l holds leaf l's box for the gap; the boxes then
      // come in as scalars, the next one while one is tested.
      auto each_leaf = [&](uint32_t child, uint32_t reach, auto&& f) {
        const uint32_t leaf0 = child * kFan, c = leaf0 + (uint32_t)lane;
        uint32_t gap = ~0u;
        if (c < t.cnt[0]) {
          const float4* b = t.box + 2ull * (t.off[0] + c);
          gap = gap_of(b[0], b[1]);
        }
        uint64_t cand = __ballot(gap <= reach);
        if (cand == 0) return;
        uint32_t j = (uint32_t)__builtin_ctzll(cand);
        const_f4 b = uniform_ptr(t.box, 2u * (t.off[0] + leaf0));
        f4v lo = b[2 * j], hi = b[2 * j + 1];
        for (;;) {
          cand &= cand - 1;
          const uint32_t jn = cand ? (uint32_t)__builtin_ctzll(cand) : j;
          const f4v nlo = b[2 * jn], nhi = b[2 * jn + 1];
          f(leaf0 + j, lane_gap(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z));
          if (cand == 0) break;
          j = jn;
          lo = nlo;
          hi = nhi;
        }
      };

      // First the leaf nearest to each query among those that meet the packet's
      // box (up to kNear of them) and its neighbours on the curve, enough
      // points for k, so that every limit is close to the final one before the
      // other leaves are chosen.
      constexpr uint32_t kFirst = KC / kLeafPts + 1;
      constexpr int kNear = 64;
      const uint32_t nfirst = min(kFirst, t.cnt[0]);
      float bestd = inf;
      uint32_t first0 = ~0u - kFirst;  // no leaf
      {
        int left = kNear;
        uint32_t best = ~0u;
        walk([] { return 0u; },
             [&](uint32_t child) {
               each_leaf(child, 0u, [&](uint32_t leaf, float d) {
                 best = d < bestd ? leaf : best;
                 bestd = fminf(bestd, d);
                 --left;
               });
               return left > 0;
             });
        if (__ballot(best != ~0u) != 0) {  // for all lanes or for none
          first0 = best - min(best, kFirst / 2);
          first0 = min(first0, t.cnt[0] - nfirst);
#pragma unroll 1
          for (uint32_t i = 0; i < nfirst; ++i) scan(first0 + i, true);
          merge();
          maxlim = wave_max_u32(lim < 0.0f ? 0u : __float_as_uint(lim));
        }
      }
      // Then the leaves within the lanes' limits.
      if constexpr (C::kOwn) {
        // Every lane queues its own, and all lanes scan one each whenever some
        // queue is full.
        uint32_t qhead = 0, qtail = 0;
        auto drain = [&](uint32_t keep) __attribute__((always_inline)) {
          while (__ballot(qtail - qhead > keep) != 0) {
            const bool on = qtail != qhead;
            const uint32_t leaf = on ? s_que[w][qhead % C::kQueue][lane] : 0u;
            qhead += on ? 1u : 0u;
            scan(leaf, on);
          }
        };
        walk([&] { return maxlim; },
             [&](uint32_t child) {
               each_leaf(child, maxlim, [&](uint32_t leaf, float d) {
                 s_que[w][qtail % C::kQueue][lane] = leaf;
                 qtail += d <= lim && leaf - first0 >= nfirst ? 1u : 0u;
                 if (__ballot(qtail - qhead == (uint32_t)C::kQueue) != 0) drain(C::kQueue / 2);
               });
               maxlim = wave_max_u32(lim < 0.0f ? 0u : __float_as_uint(lim));
               return true;
             });
        drain(0);
      } else {
        walk([&] { return maxlim; },
             [&](uint32_t child) {
               each_leaf(child, maxlim, [&](uint32_t leaf, float d) {
                 // its points are on their way while its box is tested
                 const_f4 pp = uniform_ptr(a.spts, leaf * (uint32_t)kLeafPts);
                 f4v pt[kLeafPts];
#pragma unroll
                 for (int i = 0; i < kLeafPts; ++i) pt[i] = pp[i];
                 const bool mine = leaf - first0 >= nfirst;
                 if (__ballot(d <= lim && mine) == 0) return;
#pragma unroll
                 for (int g = 0; g < kLeafPts; g += kLeafStep) {
                   room();
                   const float lm = mine ? lim : -1.0f;
#pragma unroll
                   for (int i = g; i < g + kLeafStep; ++i)
                     test(pt[i].x, pt[i].y, pt[i].z, pt[i].w, lm);
                 }
               });
               maxlim = wave_max_u32(lim < 0.0f ? 0u : __float_as_uint(lim));
               return true;
             });
      }
      merge();
    }

    if (active) {
      int32_t* oi = a.out_idx + (uint64_t)row * k;
      float* od = a.out_d2 ? a.out_d2 + (uint64_t)row * k : nullptr;
      uint32_t hits = 0;
#pragma unroll
      for (int i = 0; i < KC; ++i) {
        if ((uint32_t)i >= (uint32_t)KC - k) {
          const uint64_t key = key_bits(list[i]);
          const bool have = key < key_bits(none);
          const uint32_t j = (uint32_t)i - ((uint32_t)KC - k);
          hits += have ? 1u : 0u;
          oi[j] = have ? (int32_t)key_idx(key) : -1;
          if (od) od[j] = have ? key_d2(key) : inf;
        }
      }
      if (a.short_rows) append_short(a, hits < k && R < a.r, qs, hits, R);
    }
  }
}

template <int KC>
static void launch_kc(const SearchArgs& a, const BoxTree& t, hipStream_t st, int num_cus) {
  const uint32_t cus = (uint32_t)(num_cus > 0 ? num_cus : 256);
  const auto blocks_of = [&](uint32_t queries) {  // so many per wave
    const uint64_t per = (uint64_t)kPacketWaves * queries;
    return (uint32_t)(((uint64_t)a.nq + per - 1) / per);
  };
  const uint32_t resident = cus * (uint32_t)PacketCfg<KC>::kOccupancy;  // 4 waves a block
  const uint32_t blocks =
      a.nq_dev ? cus * 8u : std::max(blocks_of(kWave), std::min(blocks_of(1), resident));
  hipLaunchKernelGGL((k_knn_packet<KC>), dim3(blocks), dim3(kPacketWaves * kWave), 0, st, a, t);
}

hipError_t launch_knn_packet(const SearchArgs& a, const BoxTree& t, hipStream_t st, int num_cus) {
  const uint32_t k = a.k;
  if (k == 0 || k > 64 || a.tiles) return hipErrorInvalidValue;
  if (a.nq == 0) return hipSuccess;
  if (k <= 4) launch_kc<4>(a, t, st, num_cus);
  else if (k <= 8) launch_kc<8>(a, t, st, num_cus);
  else if (k <= 16) launch_kc<16>(a, t, st, num_cus);
  else if (k <= 32) launch_kc<32>(a, t, st, num_cus);
  else launch_kc<64>(a, t, st, num_cus);
  return hipGetLastError();
}

}  // namespace rtnn
