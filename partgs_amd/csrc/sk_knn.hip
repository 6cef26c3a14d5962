// Mean squared distance of every point to its three nearest neighbours:
// distCUDA2 of simple-knn (submodules/simple-knn/spatial.cu:16-27,
// simple_knn.cu:185-220), which sets the initial surfel scales of a point
// cloud (scene/gaussian_model.py:237).
//
// What is computed.  For point q, the squared distance to another point c is
// (dx dx + dy dy) + dz dz in FP32 with d = c - q (simple_knn.cu:129-133),
// each product and sum rounded on its own; the result is
// ((b0 + b1) + b2) / 3 over the three smallest such values b0 <= b1 <= b2
// (:176), FLT_MAX standing in for missing neighbours when there are fewer
// than four points (:150,162).  The reference finds them by exact search
// (its box pruning only skips boxes whose lower bound exceeds a value the
// third neighbour cannot exceed), so the result is a function of the point
// set alone; this search is exact too and returns the same bits whatever
// order it visits the points in.
//
// How.  The points are sorted by a 30-bit Morton code over their bounding
// box (whose extremes include the origin as the reference's reduction with
// init (0, 0, 0) does, :191-202) with a three-pass radix sort, and bounded by
// boxes of 16 sorted points (leaves), of 64 leaves (nodes) and of 64 nodes
// (tops).  One wave answers 64 consecutive sorted points together.  They
// search each other, then the wave's own node and the two beside it, then
// every other node whose box is within some lane's third-best.  Boxes are
// tested 64 at a time, one per lane, against the box of the lanes they
// concern; a box that passes is broadcast from its lane and each lane it
// concerns notes the leaf, and the lanes search their noted leaves together.
// 1M points on superquadrics, per call: 6.0 ms with 256-point boxes of a
// 15-bit bucket order, each box staged in LDS for a whole workgroup; 2.9 ms
// with these leaves, one wave-wide search each; 2.6 ms with per-lane lists
// (a few isolated points still had thousands of boxes tested at their first,
// wide third-best); 0.45 ms searching the neighbouring nodes first.  What is
// left is the query (0.26 ms: about 8 leaf boxes tested and 4 leaves of 16
// points searched a lane, the slowest lane of each wave bounding it) and
// sixteen short launches of the sort.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "../../include/surfel_rast.h"
#include "sr_internal.h"

namespace sk {

constexpr int kThreads = 256;
constexpr int kLeaf = 16;        // points per leaf box
constexpr int kFan = 64;         // children per node (= the wave)
constexpr int kAxisBits = 10;    // Morton bits per axis
constexpr int kDigitBits = 10;   // radix sort: bits per pass
constexpr int kPasses = 3;
constexpr int kDigits = 1 << kDigitBits;
constexpr int kItems = 16;       // keys per lane of a sorting workgroup
constexpr int kSortBlock = kThreads * kItems;
constexpr int kTodo = 6;         // leaves a lane collects before it searches them
constexpr int kMaxParts = kThreads;  // workgroups of the bounds reduction: one partial per lane when folded
static_assert(kPasses * kDigitBits == 3 * kAxisBits, "the passes cover the code");

struct Layout {
  size_t part, keys0, keys1, totals, counts, spts, boxes, nodes, tops, total;
  int nparts, nblk, nleaf, nnode, ntop;
};

inline size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

inline Layout layout(int P) {
  Layout l{};
  const size_t n = (size_t)(P > 0 ? P : 1);
  l.nparts = (int)std::min<long long>(kMaxParts, std::max<long long>(1, ((long long)P + 1023) / 1024));
  l.nblk = (int)((n + kSortBlock - 1) / kSortBlock);
  l.nleaf = (int)((n + kLeaf - 1) / kLeaf);
  l.nnode = (l.nleaf + kFan - 1) / kFan;
  l.ntop = (l.nnode + kFan - 1) / kFan;
  size_t off = 0;
  l.part = off; off += align_up((size_t)l.nparts * 6 * sizeof(float));
  l.keys0 = off; off += align_up(n * sizeof(uint2));
  l.keys1 = off; off += align_up(n * sizeof(uint2));
  l.totals = off; off += align_up((size_t)kPasses * kDigits * sizeof(uint32_t));
  l.counts = off; off += align_up((size_t)kDigits * l.nblk * sizeof(uint32_t));
  l.spts = off; off += align_up((size_t)l.nleaf * kLeaf * sizeof(float4));
  l.boxes = off; off += align_up((size_t)l.nleaf * 2 * sizeof(float4));
  l.nodes = off; off += align_up((size_t)l.nnode * 2 * sizeof(float4));
  l.tops = off; off += align_up((size_t)l.ntop * 2 * sizeof(float4));
  l.total = off;
  return l;
}

__device__ __forceinline__ float fmin_(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float fmax_(float a, float b) { return a < b ? b : a; }

// Bounding box of the points, per workgroup (grid-stride), as 6 floats.
__global__ __launch_bounds__(kThreads) void k_bounds(int P, const float* __restrict__ pts, float* part) {
  __shared__ float s[6][kThreads / 64];
  float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (int i = blockIdx.x * kThreads + threadIdx.x; i < P; i += gridDim.x * kThreads) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float v = pts[3 * (size_t)i + k];
      mn[k] = fmin_(mn[k], v);
      mx[k] = fmax_(mx[k], v);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      mn[k] = fmin_(mn[k], __shfl_xor(mn[k], off, 64));
      mx[k] = fmax_(mx[k], __shfl_xor(mx[k], off, 64));
    }
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s[k][w] = mn[k];
      s[3 + k][w] = mx[k];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    float v = s[threadIdx.x][0];
    for (int j = 1; j < kThreads / 64; ++j)
      v = threadIdx.x < 3 ? fmin_(v, s[threadIdx.x][j]) : fmax_(v, s[threadIdx.x][j]);
    part[6 * blockIdx.x + threadIdx.x] = v;
  }
}

__device__ __forceinline__ uint32_t spread10(uint32_t x) {  // 10 bits -> every third bit
  x &= 0x3ffu;
  x = (x | (x << 16)) & 0x030000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

__device__ __forceinline__ uint32_t cell_of(float v, float lo, float hi) {
  const float span = hi - lo;
  if (!(span > 0.0f)) return 0u;
  float t = (v - lo) / span * (float)(1 << kAxisBits);
  if (!(t > 0.0f)) return 0u;  // also NaN
  return t < (float)((1 << kAxisBits) - 1) ? (uint32_t)t : (uint32_t)((1 << kAxisBits) - 1);
}

// Morton code of every point, with its index.
__global__ __launch_bounds__(kThreads) void k_keys(int P, const float* __restrict__ pts, const float* part,
                                                   int nparts, uint2* keys) {
  __shared__ float s_b[6][kThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // the reference reduces with init (0, 0, 0): the origin is in the box
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    float v = (int)threadIdx.x < nparts ? part[6 * threadIdx.x + k] : 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float o = __shfl_xor(v, off, 64);
      v = k < 3 ? fmin_(v, o) : fmax_(v, o);
    }
    if (lane == 0) s_b[k][wave] = v;
  }
  __syncthreads();
  float b[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) v = k < 3 ? fmin_(v, s_b[k][w]) : fmax_(v, s_b[k][w]);
    b[k] = v;
  }
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= P) return;
  const uint32_t cx = cell_of(pts[3 * (size_t)i], b[0], b[3]);
  const uint32_t cy = cell_of(pts[3 * (size_t)i + 1], b[1], b[4]);
  const uint32_t cz = cell_of(pts[3 * (size_t)i + 2], b[2], b[5]);
  keys[i] = make_uint2(spread10(cx) | (spread10(cy) << 1) | (spread10(cz) << 2), (uint32_t)i);
}

// Radix pass, step 1: digit counts of every workgroup's kSortBlock keys
// (counts[digit][workgroup]) and over all of them (totals).
__global__ __launch_bounds__(kThreads) void k_radix_count(int P, int nblk, const uint2* __restrict__ keys, int shift,
                                                          uint32_t* counts, uint32_t* totals) {
  __shared__ uint32_t s_cnt[kDigits];
  for (int d = threadIdx.x; d < kDigits; d += kThreads) s_cnt[d] = 0u;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const long long i = (long long)blockIdx.x * kSortBlock + r * kThreads + threadIdx.x;
    if (i < P) atomicAdd(&s_cnt[(keys[i].x >> shift) & (kDigits - 1)], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kThreads) {
    const uint32_t c = s_cnt[d];
    counts[(size_t)d * nblk + blockIdx.x] = c;
    if (c) atomicAdd(&totals[d], c);
  }
}

// Step 2: one wave per digit turns its counts into the first output position
// of every workgroup's keys of that digit.
__global__ __launch_bounds__(kThreads) void k_radix_scan(int nblk, uint32_t* counts, const uint32_t* totals) {
  const int lane = threadIdx.x & 63;
  const int d = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  uint32_t base = 0;  // keys of the lower digits
#pragma unroll
  for (int t = 0; t < kDigits / 64; ++t) {
    const uint32_t c = totals[t * 64 + lane];
    base += t * 64 + lane < d ? c : 0u;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) base += (uint32_t)__shfl_xor((int)base, off, 64);
  uint32_t* row = counts + (size_t)d * nblk;
  for (int b0 = 0; b0 < nblk; b0 += 64) {
    const int b = b0 + lane;
    const uint32_t c = b < nblk ? row[b] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= off) incl += y;
    }
    if (b < nblk) row[b] = base + incl - c;
    base += (uint32_t)__shfl((int)incl, 63, 64);
  }
}

// Step 3: stable scatter.  Wave w of a workgroup owns the w-th quarter of
// its keys and places them 64 at a time in order; lanes of the same digit
// find each other by ballots.  kLast: the points themselves are written
// (x, y, z, index bits) instead of the keys.
template <bool kLast>
__global__ __launch_bounds__(kThreads) void k_radix_scatter(int P, int nblk, const uint2* __restrict__ keys, int shift,
                                                            const uint32_t* __restrict__ counts, uint2* out,
                                                            const float* __restrict__ pts, float4* spts) {
  constexpr int kWaves = kThreads / 64;
  __shared__ uint32_t s_at[kWaves][kDigits];  // next output position per (wave, digit)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int d = threadIdx.x; d < kWaves * kDigits; d += kThreads) (&s_at[0][0])[d] = 0u;
  __syncthreads();
  const long long first = (long long)blockIdx.x * kSortBlock + wave * (64 * kItems) + lane;
  uint2 kv[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) kv[r] = first + r * 64 < P ? keys[first + r * 64] : make_uint2(0u, 0u);
#pragma unroll
  for (int r = 0; r < kItems; ++r)
    if (first + r * 64 < P) atomicAdd(&s_at[wave][(kv[r].x >> shift) & (kDigits - 1)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kThreads) {
    uint32_t at = counts[(size_t)d * nblk + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t c = s_at[w][d];
      s_at[w][d] = at;
      at += c;
    }
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const bool in = first + r * 64 < P;
    const uint32_t d = (kv[r].x >> shift) & (kDigits - 1);
    uint64_t same = __ballot(in);
#pragma unroll
    for (int t = 0; t < kDigitBits; ++t) {
      const bool bit = (d >> t) & 1u;
      const uint64_t m = __ballot(bit);
      same &= bit ? m : ~m;
    }
    const int leader = same ? __builtin_ctzll(same) : lane;
    uint32_t at = 0;
    if (in && lane == leader) at = atomicAdd(&s_at[wave][d], (uint32_t)__popcll(same));
    at = (uint32_t)__shfl((int)at, leader, 64) + (uint32_t)__popcll(same & below);
    if (in) {
      if (kLast) {
        const size_t i = kv[r].y;
        spts[at] = make_float4(pts[3 * i], pts[3 * i + 1], pts[3 * i + 2], __uint_as_float(kv[r].y));
      } else {
        out[at] = kv[r];
      }
    }
  }
}

struct Bounds {
  float4 lo, hi;
};
__device__ __forceinline__ Bounds no_bounds() {
  return {make_float4(FLT_MAX, FLT_MAX, FLT_MAX, 0.0f), make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, 0.0f)};
}
// Union with the lane `off` away.
__device__ __forceinline__ void merge_xor(Bounds& b, int off) {
  b.lo.x = fmin_(b.lo.x, __shfl_xor(b.lo.x, off, 64));
  b.lo.y = fmin_(b.lo.y, __shfl_xor(b.lo.y, off, 64));
  b.lo.z = fmin_(b.lo.z, __shfl_xor(b.lo.z, off, 64));
  b.hi.x = fmax_(b.hi.x, __shfl_xor(b.hi.x, off, 64));
  b.hi.y = fmax_(b.hi.y, __shfl_xor(b.hi.y, off, 64));
  b.hi.z = fmax_(b.hi.z, __shfl_xor(b.hi.z, off, 64));
}
__device__ __forceinline__ void add_point(Bounds& b, const float4& p) {
  b.lo.x = fmin_(b.lo.x, p.x);
  b.lo.y = fmin_(b.lo.y, p.y);
  b.lo.z = fmin_(b.lo.z, p.z);
  b.hi.x = fmax_(b.hi.x, p.x);
  b.hi.y = fmax_(b.hi.y, p.y);
  b.hi.z = fmax_(b.hi.z, p.z);
}

// Leaf boxes, one lane per point.  The last leaf is filled up with NaN
// points, which are nobody's neighbour.
__global__ __launch_bounds__(kThreads) void k_boxes(int P, int nleaf, float4* spts, float4* boxes) {
  const long long i = (long long)blockIdx.x * kThreads + threadIdx.x;
  Bounds b = no_bounds();
  if (i < P) {
    add_point(b, spts[i]);
  } else if (i < (long long)nleaf * kLeaf) {
    const float nan = __builtin_nanf("");
    spts[i] = make_float4(nan, nan, nan, 0.0f);
  }
#pragma unroll
  for (int off = kLeaf / 2; off > 0; off >>= 1) merge_xor(b, off);
  if (i < P && threadIdx.x % kLeaf == 0) {
    boxes[2 * (i / kLeaf)] = b.lo;
    boxes[2 * (i / kLeaf) + 1] = b.hi;
  }
}

// Bounds of every kFan consecutive boxes, one wave each.
__global__ __launch_bounds__(64) void k_groups(int nbox, const float4* __restrict__ boxes, float4* groups) {
  const int i = blockIdx.x * kFan + (int)threadIdx.x;
  Bounds b = no_bounds();
  if (i < nbox) {
    b.lo = boxes[2 * i];
    b.hi = boxes[2 * i + 1];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) merge_xor(b, off);
  if (threadIdx.x == 0) {
    groups[2 * blockIdx.x] = b.lo;
    groups[2 * blockIdx.x + 1] = b.hi;
  }
}

// distBoxPoint, simple_knn.cu:115-125: a lower bound of the squared
// distance from p to any point inside the box.
__device__ __forceinline__ float box_dist(const float4& lo, const float4& hi, float px, float py, float pz) {
  float dx = 0.0f, dy = 0.0f, dz = 0.0f;
  if (px < lo.x || px > hi.x) dx = fmin_(fabsf(px - lo.x), fabsf(px - hi.x));
  if (py < lo.y || py > hi.y) dy = fmin_(fabsf(py - lo.y), fabsf(py - hi.y));
  if (pz < lo.z || pz > hi.z) dz = fmin_(fabsf(pz - lo.z), fabsf(pz - hi.z));
  return dx * dx + dy * dy + dz * dz;
}

// Lower bound of the squared distance between points of two boxes.  Every
// step rounds monotonically, so in FP32 it is at most box_dist of any point
// of one box to the other, which is at most the distance itself.
__device__ __forceinline__ float box_box(const Bounds& a, const float4& lo, const float4& hi) {
  const float dx = fmax_(0.0f, fmax_(lo.x - a.hi.x, a.lo.x - hi.x));
  const float dy = fmax_(0.0f, fmax_(lo.y - a.hi.y, a.lo.y - hi.y));
  const float dz = fmax_(0.0f, fmax_(lo.z - a.hi.z, a.lo.z - hi.z));
  return dx * dx + dy * dy + dz * dz;
}

// updateKBest<3>, simple_knn.cu:127-143: insertion into the ascending triple
// (b0 <= b1 <= b2: the new ones are the minimum and two medians).  A NaN or
// infinite distance enters as FLT_MAX, which is no neighbour.
__device__ __forceinline__ void update_best(float px, float py, float pz, const float4& c, bool self, float* best) {
  const float dx = c.x - px, dy = c.y - py, dz = c.z - pz;
  float d = fminf(dx * dx + dy * dy + dz * dz, FLT_MAX);
  d = self ? FLT_MAX : d;
  best[2] = __builtin_amdgcn_fmed3f(best[1], best[2], d);
  best[1] = __builtin_amdgcn_fmed3f(best[0], best[1], d);
  best[0] = fminf(best[0], d);
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__global__ __launch_bounds__(kThreads) void k_query(int P, int nleaf, int nnode, int ntop,
                                                    const float4* __restrict__ spts,
                                                    const float4* __restrict__ boxes,
                                                    const float4* __restrict__ nodes,
                                                    const float4* __restrict__ tops, float* out) {
  __shared__ uint2 s_todo[kThreads / 64][kTodo][64];  // per lane: (leaf, its box's distance) still to search
  const int lane = threadIdx.x & 63;
  const int grp = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)));
  const int p0 = grp * 64;
  if (p0 >= P) return;
  uint2(*todo)[64] = s_todo[threadIdx.x >> 6];
  int ntodo = 0;
  const int pos = p0 + lane;
  const bool valid = pos < P;
  const float4 q = spts[min(pos, P - 1)];
  // a NaN coordinate is at no finite distance from anything
  const bool ask = valid && q.x == q.x && q.y == q.y && q.z == q.z;
  float best[3] = {FLT_MAX, FLT_MAX, FLT_MAX};
  const int own = min(64, P - p0);
  for (int k = 0; k < own; ++k) {
    const float4 c = make_float4(lane_value(q.x, k), lane_value(q.y, k), lane_value(q.z, k), 0.0f);
    update_best(q.x, q.y, q.z, c, k == lane, best);
  }
  const int own_leaf = p0 / kLeaf, own_node = own_leaf / kFan;
  // every lane searches the leaves on its list that are still near enough
  auto search = [&]() {
    for (int t = 0; __ballot(t < ntodo) != 0ull; ++t) {
      if (t >= ntodo) continue;
      const uint2 e = todo[t][lane];
      if (__uint_as_float(e.y) > best[2]) continue;
      const float4* c = spts + (size_t)e.x * kLeaf;
      float4 v[kLeaf];
#pragma unroll
      for (int k = 0; k < kLeaf; ++k) v[k] = c[k];
#pragma unroll
      for (int k = 0; k < kLeaf; ++k) update_best(q.x, q.y, q.z, v[k], false, best);
    }
    ntodo = 0;
  };
  // bit i: box i of the kFan from b0 on comes within the worst third-best of
  // the lanes with `in` set of those lanes' own box; mine receives this
  // lane's box
  auto near = [&](const float4* b, int b0, int n, bool in, Bounds& mine) -> uint64_t {
    Bounds g = no_bounds();
    if (in) add_point(g, q);
    float worst = in ? best[2] : 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      merge_xor(g, off);
      worst = fmax_(worst, __shfl_xor(worst, off, 64));
    }
    const int i = b0 + lane;
    bool hit = false;
    if (i < n) {
      mine.lo = b[2 * i];
      mine.hi = b[2 * i + 1];
      hit = !(box_box(g, mine.lo, mine.hi) > worst);
    }
    return __ballot(hit);
  };
  // box j of a batch (lane j holds it) against this lane's point
  auto dist_to = [&](const Bounds& b, int j) {
    const float4 lo = make_float4(lane_value(b.lo.x, j), lane_value(b.lo.y, j), lane_value(b.lo.z, j), 0.0f);
    const float4 hi = make_float4(lane_value(b.hi.x, j), lane_value(b.hi.y, j), lane_value(b.hi.z, j), 0.0f);
    return box_dist(lo, hi, q.x, q.y, q.z);
  };
  // puts a node's leaves on the lists of the lanes they concern; need: the
  // lanes the node's box concerns
  auto visit = [&](int node, bool need) {
    if (__ballot(need) == 0ull) return;
    const int l0 = node * kFan;
    Bounds bx = no_bounds();
    uint64_t ml = near(boxes, l0, nleaf, need, bx);
    for (; ml; ml &= ml - 1ull) {
      const int j = __builtin_ctzll(ml), leaf = l0 + j;
      if (leaf >= own_leaf && leaf < own_leaf + 64 / kLeaf) continue;
      const float d = dist_to(bx, j);
      if (need && !(d > best[2])) todo[ntodo++][lane] = make_uint2((uint32_t)leaf, __float_as_uint(d));
      if (__ballot(ntodo == kTodo) != 0ull) search();
    }
  };
  // the wave's own node and the two beside it first: what is near along the
  // curve leaves few lanes with anything left to find elsewhere
  const int w0 = max(own_node - 1, 0), w1 = min(own_node + 1, nnode - 1);
  for (int t = 0; t < 3; ++t) {
    const int node = own_node + (t == 0 ? 0 : (t == 1 ? -1 : 1));
    if (node < w0 || node > w1) continue;
    visit(node, ask && !(box_dist(nodes[2 * node], nodes[2 * node + 1], q.x, q.y, q.z) > best[2]));
  }
  search();
  for (int t0 = 0; t0 < ntop; t0 += kFan) {
    Bounds bt = no_bounds();
    uint64_t mt = near(tops, t0, ntop, ask, bt);
    for (; mt; mt &= mt - 1ull) {
      const int jt = __builtin_ctzll(mt), n0 = (t0 + jt) * kFan;
      const bool want = ask && !(dist_to(bt, jt) > best[2]);
      if (__ballot(want) == 0ull) continue;
      Bounds bn = no_bounds();
      uint64_t mn = near(nodes, n0, nnode, want, bn);
      for (; mn; mn &= mn - 1ull) {
        const int jn = __builtin_ctzll(mn), node = n0 + jn;
        if (node >= w0 && node <= w1) continue;
        visit(node, want && !(dist_to(bn, jn) > best[2]));
      }
    }
  }
  search();
  if (valid) out[__float_as_uint(q.w)] = (best[0] + best[1] + best[2]) / 3.0f;
}

__global__ void k_zero(uint32_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

}  // namespace sk

extern "C" {

size_t sk_dist2_workspace_bytes(int P) {
  if (P < 0) return 0;
  return sk::layout(P).total;
}

int sk_dist2(int P, const float* points, float* mean_dists, void* workspace, size_t workspace_bytes,
             sr_stream_t stream) {
  if (P < 0) return sr::set_error(SR_ERR_INVALID, "sk_dist2: P must be >= 0");
  if (P == 0) return SR_OK;
  if (!points || !mean_dists) return sr::set_error(SR_ERR_INVALID, "sk_dist2: NULL points or output");
  if (P > (1 << 30)) return sr::set_error(SR_ERR_INVALID, "sk_dist2: more than 2^30 points");
  const sk::Layout l = sk::layout(P);
  if (!workspace || workspace_bytes < l.total)
    return sr::set_error(SR_ERR_INVALID, "sk_dist2: workspace smaller than sk_dist2_workspace_bytes(P)");
  char* ws = (char*)workspace;
  float* part = (float*)(ws + l.part);
  uint2* k0 = (uint2*)(ws + l.keys0);
  uint2* k1 = (uint2*)(ws + l.keys1);
  uint32_t* totals = (uint32_t*)(ws + l.totals);
  uint32_t* counts = (uint32_t*)(ws + l.counts);
  float4* spts = (float4*)(ws + l.spts);
  float4* boxes = (float4*)(ws + l.boxes);
  float4* nodes = (float4*)(ws + l.nodes);
  float4* tops = (float4*)(ws + l.tops);
  hipStream_t s = (hipStream_t)stream;
  const dim3 th(sk::kThreads);
  const unsigned pb = (unsigned)(((long long)P + sk::kThreads - 1) / sk::kThreads);
  const int nt = sk::kPasses * sk::kDigits;
  hipLaunchKernelGGL(sk::k_zero, dim3((nt + 255) / 256), dim3(256), 0, s, totals, nt);
  hipLaunchKernelGGL(sk::k_bounds, dim3(l.nparts), th, 0, s, P, points, part);
  hipLaunchKernelGGL(sk::k_keys, dim3(pb), th, 0, s, P, points, part, l.nparts, k0);
  for (int pass = 0; pass < sk::kPasses; ++pass) {
    const int shift = pass * sk::kDigitBits;
    hipLaunchKernelGGL(sk::k_radix_count, dim3(l.nblk), th, 0, s, P, l.nblk, k0, shift, counts,
                       totals + pass * sk::kDigits);
    hipLaunchKernelGGL(sk::k_radix_scan, dim3(sk::kDigits / (sk::kThreads / 64)), th, 0, s, l.nblk, counts,
                       totals + pass * sk::kDigits);
    if (pass + 1 < sk::kPasses)
      hipLaunchKernelGGL(sk::k_radix_scatter<false>, dim3(l.nblk), th, 0, s, P, l.nblk, k0, shift, counts, k1, points,
                         spts);
    else
      hipLaunchKernelGGL(sk::k_radix_scatter<true>, dim3(l.nblk), th, 0, s, P, l.nblk, k0, shift, counts, k1, points,
                         spts);
    std::swap(k0, k1);
  }
  hipLaunchKernelGGL(sk::k_boxes, dim3(pb), th, 0, s, P, l.nleaf, spts, boxes);
  hipLaunchKernelGGL(sk::k_groups, dim3(l.nnode), dim3(64), 0, s, l.nleaf, boxes, nodes);
  hipLaunchKernelGGL(sk::k_groups, dim3(l.ntop), dim3(64), 0, s, l.nnode, nodes, tops);
  hipLaunchKernelGGL(sk::k_query, dim3(pb), th, 0, s, P, l.nleaf, l.nnode, l.ntop, spts, boxes, nodes, tops,
                     mean_dists);
  return hipGetLastError() == hipSuccess ? SR_OK : sr::set_error(SR_ERR_HIP, "sk_dist2: kernel launch failed");
}

}  // extern "C"
