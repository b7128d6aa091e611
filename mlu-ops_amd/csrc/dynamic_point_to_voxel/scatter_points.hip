// Dynamic point-to-voxel scatter, forward: points that share a coordinate
// triple form a voxel; voxels are numbered in ascending (lexicographic) order
// of their triples; the features of a voxel's points are reduced by max or
// mean.  The reference delegates the grouping to a vendor "unique" routine
// (kernels/dynamic_point_to_voxel/dynamic_point_to_voxel_forward/
//  dynamic_point_to_voxel_forward.cpp:300-340) and reduces with atomics.
//
// Here:
//   1 dpvPrepare, dpvAxisMax  rows with a negative coordinate become (-1,-1,-1) in place; the largest
//                  coordinate of every axis goes to the host, so that the sorts run over as few
//                  bits as the data needs
//   2 one stable radix sort of (packed triple, point index): 64-bit records of both when the triples,
//                  numbered in mixed radix, fit 32 bits; pairs when the three coordinates (+1) fit
//                  64 bits together; otherwise three stable sorts, last axis first.  Either way the
//                  points end up in ascending triple order, equal triples in point order
//   3 rankFlags    bitmap of the sorted positions where a triple starts, with prefix sums
//   4 dpvEmit      point2voxel_map, voxel_coors, first sorted position of
//                  every voxel, voxel_num
//   5 dpvReduce    up to four features of a voxel a thread, which walks the voxel's points in
//                  point order: max, or the sum of feats / count in exactly
//                  the order the sequential definition adds them, so the mean
//                  has the same bits on every run; rows without a voxel get their fill here as well
//
// What bounds it: rows of features read and written at random places (dpvReduce moves 100 MB in 32 us
// at 400 k points of 32 features), and launches that each start cold, the sort's nine most of all.
// Measured there: 105 us forward, 72 us backward; 165 and 88 us with four passes of 8 bits, separate
// fills, one feature a thread and atomic minima.
#include <hip/hip_runtime.h>

#include <initializer_list>

#include "core/core.h"
#include "core/device_sort.h"

#include "dynamic_point_to_voxel/scatter_points.h"

namespace mluop {
namespace dynamic_point_to_voxel {
namespace {

using device_sort::u64;

constexpr int kBlock = device_sort::kFlagThreads;
constexpr int kPrepareBlocks = 512;

inline int gridFor(size_t n, int cap = 1 << 30) {
  size_t b = (n + kBlock - 1) / kBlock;
  if (b < 1) b = 1;
  return (int)(b > (size_t)cap ? (size_t)cap : b);
}

size_t alignUp(size_t v) { return (v + 255) & ~(size_t)255; }

// Negative rows masked; the block's largest coordinates to block_max[axis][block].
__global__ __launch_bounds__(kBlock) void dpvPrepare(int32_t *coors, int n, int32_t *block_max) {
  int m0 = -1, m1 = -1, m2 = -1;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    int c0 = coors[3 * (size_t)i];
    int c1 = coors[3 * (size_t)i + 1];
    int c2 = coors[3 * (size_t)i + 2];
    if (c0 < 0 || c1 < 0 || c2 < 0) {
      c0 = c1 = c2 = -1;
      coors[3 * (size_t)i] = -1;
      coors[3 * (size_t)i + 1] = -1;
      coors[3 * (size_t)i + 2] = -1;
    }
    m0 = max(m0, c0);
    m1 = max(m1, c1);
    m2 = max(m2, c2);
  }
  __shared__ int s_max[3][kBlock / 64];
  for (int off = 32; off > 0; off >>= 1) {
    m0 = max(m0, __shfl_xor(m0, off, 64));
    m1 = max(m1, __shfl_xor(m1, off, 64));
    m2 = max(m2, __shfl_xor(m2, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    s_max[0][threadIdx.x >> 6] = m0;
    s_max[1][threadIdx.x >> 6] = m1;
    s_max[2][threadIdx.x >> 6] = m2;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    int m = s_max[threadIdx.x][0];
    for (int w = 1; w < kBlock / 64; ++w) m = max(m, s_max[threadIdx.x][w]);
    block_max[threadIdx.x * kPrepareBlocks + blockIdx.x] = m;
  }
}

// A wave per axis; the result goes to the host, below the low half of the stamp.
__global__ __launch_bounds__(192) void dpvAxisMax(const int32_t *__restrict__ block_max, int blocks, u64 *host_words,
                                                  u64 stamp) {
  const int axis = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int m = -1;
  for (int b = lane; b < blocks; b += 64) m = max(m, block_max[axis * kPrepareBlocks + b]);
  for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
  if (lane == 0)
    __hip_atomic_store(host_words + axis, stamp << 32 | (uint32_t)m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Triples (c0+1, c1+1, c2+1) numbered in mixed radix (rows are masked already: 0 is the -1 triple).
struct TripleRadix {
  uint32_t d1, d2;  // values of the last two axes
  __device__ uint32_t number(const int32_t *c) const {
    return ((uint32_t)(c[0] + 1) * d1 + (uint32_t)(c[1] + 1)) * d2 + (uint32_t)(c[2] + 1);
  }
  __device__ void coordinates(uint32_t number, int32_t *c) const {
    const uint32_t rest = number / d2;
    c[2] = (int32_t)(number - rest * d2) - 1;
    const uint32_t first = rest / d1;
    c[1] = (int32_t)(rest - first * d1) - 1;
    c[0] = (int32_t)first - 1;
  }
};

// First pass of the sort of records (triple number in the low half, point index in the high half:
// sorted as one key by the low bits, the point travels with it), straight from the coordinates.
struct RecordsOfPoints {
  typedef uint32_t Item;
  const int32_t *coors;
  TripleRadix radix;
  uint32_t mask;
  u64 *records;
  __device__ Item load(int64_t i) const { return radix.number(coors + 3 * i); }
  __device__ uint32_t digit(Item t) const { return t & mask; }
  __device__ void store(size_t to, Item t, int64_t i) const { records[to] = (u64)i << 32 | t; }
};

// key = (c0+1, c1+1, c2+1) packed most significant first; rows are already masked
__global__ __launch_bounds__(kBlock) void dpvPackKeys(const int32_t *__restrict__ coors, int n, int bits1, int bits2,
                                                      u64 *__restrict__ keys, uint32_t *__restrict__ points) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const u64 k0 = (uint32_t)(coors[3 * (size_t)i] + 1);
  const u64 k1 = (uint32_t)(coors[3 * (size_t)i + 1] + 1);
  const u64 k2 = (uint32_t)(coors[3 * (size_t)i + 2] + 1);
  keys[i] = (k0 << (bits1 + bits2)) | (k1 << bits2) | k2;
  points[i] = (uint32_t)i;
}

// keys[p] = coordinate `axis` of the point at position p, plus one (`first`: the points in their order,
// which are written as well)
__global__ __launch_bounds__(kBlock) void dpvAxisKeys(const int32_t *__restrict__ coors, uint32_t *points, bool first,
                                                      int n, int axis, uint32_t *__restrict__ keys) {
  const int p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= n) return;
  const uint32_t i = first ? (uint32_t)p : points[p];
  if (first) points[p] = i;
  keys[p] = (uint32_t)(coors[3 * (size_t)i + axis] + 1);
}

// The sorted points: in the high halves of records, or by themselves.
struct SortedPoints {
  const u64 *records;
  const uint32_t *points;
  __device__ uint32_t at(int64_t p) const { return records != nullptr ? (uint32_t)(records[p] >> 32) : points[p]; }
};

// Positions where the triple differs from the one in front.
template <bool RECORDS>
struct TripleStarts {
  SortedPoints sorted;
  const int32_t *coors;
  __device__ bool flagged(int64_t p) const {
    const int64_t q = p > 0 ? p - 1 : 0;
    if (RECORDS)
      return ((uint32_t)sorted.records[p] != (uint32_t)sorted.records[q]) | (p == 0);
    const int32_t *a = coors + 3 * (size_t)sorted.points[p];
    const int32_t *b = coors + 3 * (size_t)sorted.points[q];
    return (a[0] != b[0]) | (a[1] != b[1]) | (a[2] != b[2]) | (p == 0);
  }
};

__global__ __launch_bounds__(kBlock) void dpvEmit(const int32_t *__restrict__ coors, SortedPoints sorted,
                                                  TripleRadix radix, device_sort::FlagRanks starts, int n, int rows,
                                                  int32_t *__restrict__ point2voxel_map,
                                                  int32_t *__restrict__ voxel_coors, int32_t *__restrict__ first_pos,
                                                  int32_t *__restrict__ voxel_num) {
  __shared__ device_sort::FlagSums s_sums;
  const int p = blockIdx.x * kBlock + threadIdx.x;
  s_sums.add(starts);
  if (p >= n) return;
  // the (-1,-1,-1) triple sorts first and is not a voxel
  const int skipped = coors[3 * (size_t)sorted.at(0)] == -1 ? 1 : 0;
  const bool head = device_sort::FlagSums::flagged(starts, p);
  const int v = (int)s_sums.before(starts, p) - (head ? 0 : 1) - skipped;
  const uint32_t i = sorted.at(p);
  point2voxel_map[i] = v;
  if (head && v >= 0 && v <= rows) {
    first_pos[v] = p;  // one past the last stored voxel included: it ends that voxel
    if (v < rows) {
      int32_t c[3] = {0, 0, 0};
      if (sorted.records != nullptr) {
        radix.coordinates((uint32_t)sorted.records[p], c);
      } else {
        for (int a = 0; a < 3; ++a) c[a] = coors[3 * (size_t)i + a];
      }
      for (int a = 0; a < 3; ++a) voxel_coors[3 * (size_t)v + a] = c[a];
    }
  }
  if (p == n - 1) *voxel_num = v + 1;
}

template <int VEC>
struct alignas(4 * VEC) Floats {
  float x[VEC];
};

// Thread t takes VEC features of row t / (C / VEC).  Points of a voxel are read four ahead of the
// reduction, which keeps their order.
template <int VEC, bool MAX>
__global__ __launch_bounds__(kBlock) void dpvReduce(const float *__restrict__ feats, SortedPoints sorted,
                                                    const int32_t *__restrict__ first_pos,
                                                    const int32_t *__restrict__ voxel_num, int n, int num_features,
                                                    int rows, float *__restrict__ voxel_feats,
                                                    int32_t *__restrict__ voxel_coors,
                                                    int32_t *__restrict__ voxel_points_count) {
  constexpr int kAhead = 4;
  typedef Floats<VEC> F;
  const uint32_t lanes = (uint32_t)num_features / VEC;
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;  // (fewer than 2^31 features in all)
  const uint32_t v = t / lanes;
  if (v >= (uint32_t)rows) return;
  const int f = (int)(t - v * lanes) * VEC;
  F *out = reinterpret_cast<F *>(voxel_feats + (size_t)v * num_features + f);
  F acc;
#pragma unroll
  for (int k = 0; k < VEC; ++k) acc.x[k] = MAX ? -INFINITY : 0.f;
  const int voxels = *voxel_num;
  if (v >= (uint32_t)voxels) {
    *out = acc;
    if (f == 0) {
      voxel_points_count[v] = 0;
      for (int a = 0; a < 3; ++a) voxel_coors[3 * (size_t)v + a] = 0;
    }
    return;
  }
  const int begin = first_pos[v];
  // dpvEmit stores the first position of voxel `rows` too, when there is one
  const int stop = (int)v + 1 < voxels ? first_pos[v + 1] : n;
  const int count = stop - begin;
  if (f == 0) voxel_points_count[v] = count;
  const float fcount = (float)count;
  for (int p = begin; p < stop; p += kAhead) {
    F x[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      x[u] = *reinterpret_cast<const F *>(feats + (size_t)sorted.at(min(p + u, stop - 1)) * num_features + f);
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (p + u < stop) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          if (MAX)
            acc.x[k] = x[u].x[k] >= acc.x[k] ? x[u].x[k] : acc.x[k];
          else
            acc.x[k] = __fadd_rn(acc.x[k], __fdiv_rn(x[u].x[k], fcount));
        }
      }
  }
  *out = acc;
}

// ---- backward of the max reduction ----
//
// The gradient of (voxel, feature) goes to the lowest point whose feature equals the maximum.
// Rows of many features: the points of every voxel are listed first, in any order; then the threads
// of a voxel go through its points once, reading and writing every row once.  A voxel of more than
// kListed points has no list, and no thread walks it: its points look for themselves, with an
// atomic minimum for every feature that equals the maximum, and write their rows in a launch of
// their own, which finds nothing to do where there is no such voxel.  Where voxels have more points
// than that on average nothing is listed at all.
// Rows of few features: the atomic minimum for every point (see below), which needs no lists.

__device__ inline bool inVoxel(int v, const int32_t *voxel_num, int rows) { return v >= 0 && v < min(*voxel_num, rows); }

constexpr uint32_t kListed = 32;              // points of a voxel that has a list
constexpr uint32_t kUnlisted = 0x80000000u;   // starts[v]: this and the number of the voxel among those without one

// So few voxels that each can go without a list (`unlisted_most` of them can).
__device__ inline bool nothingListed(int voxels, uint32_t unlisted_most) { return voxels <= (int)unlisted_most; }

// What the launches hand on beside the arrays, in device memory.
struct ListTotals {
  uint32_t listed;    // points in lists
  uint32_t unlisted;  // voxels without one
};

__global__ __launch_bounds__(kBlock) void dpvBackwardClearCounts(uint32_t *counts, int rows, ListTotals *totals) {
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < rows) counts[v] = 0;
  if (v == 0) *totals = ListTotals{0, 0};
}

// counts[v] = points of voxel v, arrival[x] = points of its voxel counted before point x.  The points
// of a workgroup are counted in LDS first, so that a voxel costs one atomic a workgroup however many
// of its points are there (atomics on one word take 11 ns each).
constexpr int kCountThreads = 512;
constexpr int kCountPer = 4;
constexpr int kCountSlots = 2 * kCountThreads * kCountPer;
__global__ __launch_bounds__(kCountThreads) void dpvBackwardCount(const int32_t *__restrict__ point2voxel_map,
                                                                  const int32_t *__restrict__ voxel_num, int n,
                                                                  int rows, uint32_t unlisted_most, uint32_t *counts,
                                                                  uint32_t *__restrict__ arrival) {
  __shared__ uint32_t s_voxel[kCountSlots], s_count[kCountSlots];
  constexpr uint32_t kEmpty = 0xffffffffu;
  const int tid = threadIdx.x;
  const int first = blockIdx.x * (kCountThreads * kCountPer) + tid;
  const int voxels = min(*voxel_num, rows);
  if (nothingListed(voxels, unlisted_most)) return;
  int v[kCountPer];
#pragma unroll
  for (int u = 0; u < kCountPer; ++u) {
    const int x = first + u * kCountThreads;
    v[u] = x < n ? point2voxel_map[x] : -1;
  }
  for (int s = tid; s < kCountSlots; s += kCountThreads) {
    s_voxel[s] = kEmpty;
    s_count[s] = 0;
  }
  __syncthreads();
  uint32_t slot[kCountPer], before[kCountPer];
#pragma unroll
  for (int u = 0; u < kCountPer; ++u) {
    if (v[u] >= voxels) v[u] = -1;
    if (v[u] < 0) continue;
    uint32_t at = ((uint32_t)v[u] * 0x9e3779b1u) / (0xffffffffu / kCountSlots + 1);
    // (twice as many slots as points: an empty one is always reached)
    while (true) {
      const uint32_t seen = atomicCAS(&s_voxel[at], kEmpty, (uint32_t)v[u]);
      if (seen == kEmpty || seen == (uint32_t)v[u]) break;
      at = (at + 1) & (kCountSlots - 1);
    }
    slot[u] = at;
    before[u] = atomicAdd(&s_count[at], 1u);
  }
  __syncthreads();
  for (int s = tid; s < kCountSlots; s += kCountThreads)
    if (s_voxel[s] != kEmpty) s_count[s] = atomicAdd(&counts[s_voxel[s]], s_count[s]);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kCountPer; ++u)
    if (v[u] >= 0) arrival[first + u * kCountThreads] = s_count[slot[u]] + before[u];
}

// starts[v] = where the list of voxel v starts (the lists lie in no particular order: one atomic a
// workgroup hands out the space, 8 ns each since they all go to one word), or its number among the
// voxels without one.
constexpr int kPlaceThreads = 1024;
constexpr int kPlacePer = 4;
__global__ __launch_bounds__(kPlaceThreads) void dpvBackwardPlaces(const uint32_t *__restrict__ counts,
                                                                   const int32_t *__restrict__ voxel_num, int rows,
                                                                   uint32_t unlisted_most, ListTotals *totals,
                                                                   uint32_t *__restrict__ starts) {
  // a workgroup's points in lists, and above them its voxels without one
  constexpr int kShift = 18;
  static_assert(kPlaceThreads * kPlacePer * kListed < 1u << kShift && kPlaceThreads * kPlacePer < 1 << (32 - kShift),
                "both sums in one word");
  __shared__ uint32_t s_wave[kPlaceThreads / 64];
  __shared__ uint32_t s_listed, s_unlisted;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int first = (blockIdx.x * kPlaceThreads + tid) * kPlacePer;
  const int voxels = min(*voxel_num, rows);
  if (nothingListed(voxels, unlisted_most)) {
    for (int u = 0; u < kPlacePer; ++u)
      if (first + u < rows) starts[first + u] = kUnlisted | (uint32_t)(first + u);
    if (first == 0) totals->unlisted = (uint32_t)max(voxels, 0);
    return;
  }
  uint32_t c[kPlacePer], sum = 0;
#pragma unroll
  for (int u = 0; u < kPlacePer; ++u) {
    c[u] = first + u < rows ? counts[first + u] : 0u;
    if (c[u] > kListed) c[u] = 1u << kShift;
    sum += c[u];
  }
  const uint32_t incl = device_sort::waveInclusiveSum(sum);
  if ((tid & 63) == 63) s_wave[wave] = incl;
  __syncthreads();
  if (tid == 0) {
    uint32_t all = 0;
    for (int w = 0; w < kPlaceThreads / 64; ++w) all += s_wave[w];
    const uint32_t listed = all & ((1u << kShift) - 1u), unlisted = all >> kShift;
    s_listed = listed == 0 ? 0u : atomicAdd(&totals->listed, listed);
    s_unlisted = unlisted == 0 ? 0u : atomicAdd(&totals->unlisted, unlisted);
  }
  __syncthreads();
  uint32_t in_front = incl - sum;
  for (int w = 0; w < wave; ++w) in_front += s_wave[w];
#pragma unroll
  for (int u = 0; u < kPlacePer; ++u) {
    if (first + u < rows)
      starts[first + u] = c[u] >> kShift != 0 ? kUnlisted | (s_unlisted + (in_front >> kShift))
                                              : s_listed + (in_front & ((1u << kShift) - 1u));
    in_front += c[u];
  }
}

// The first `list_blocks` workgroups write the lists, the others from[voxel without a list, feature] = n.
__global__ __launch_bounds__(kBlock) void dpvBackwardList(const int32_t *__restrict__ point2voxel_map,
                                                          const int32_t *__restrict__ voxel_num, int n, int rows,
                                                          int num_features, int list_blocks,
                                                          const uint32_t *__restrict__ starts,
                                                          const uint32_t *__restrict__ arrival,
                                                          uint32_t *__restrict__ points,
                                                          const ListTotals *__restrict__ totals,
                                                          int32_t *__restrict__ from) {
  if ((int)blockIdx.x >= list_blocks) {
    const size_t words = (size_t)totals->unlisted * num_features;
    for (size_t i = (size_t)(blockIdx.x - list_blocks) * kBlock + threadIdx.x; i < words;
         i += (size_t)(gridDim.x - list_blocks) * kBlock)
      from[i] = n;
    return;
  }
  const int x = blockIdx.x * kBlock + threadIdx.x;
  if (x >= n) return;
  const int v = point2voxel_map[x];
  if (!inVoxel(v, voxel_num, rows)) return;
  const uint32_t start = starts[v];
  if ((start & kUnlisted) == 0) points[start + arrival[x]] = (uint32_t)x;
}

// Thread t takes VEC features of the listed voxel t / (C / VEC), and of the point of that number if it
// is in no voxel or in one without a list.  Up to four points of a voxel are held at once and their
// rows written whole.
template <int VEC>
__global__ __launch_bounds__(kBlock) void dpvBackwardVoxels(
    const float *__restrict__ grad_voxel_feats, const float *__restrict__ feats,
    const float *__restrict__ voxel_feats, const int32_t *__restrict__ point2voxel_map,
    const int32_t *__restrict__ voxel_num, int n, int num_features, int rows, const uint32_t *__restrict__ counts,
    const uint32_t *__restrict__ starts, const uint32_t *__restrict__ points, int32_t *from, float *grad_feats) {
  typedef Floats<VEC> F;
  constexpr int kHeld = 4;
  const uint32_t lanes = (uint32_t)num_features / VEC;
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;  // (fewer than 2^31 features in all)
  const uint32_t v = t / lanes;
  if (v >= (uint32_t)n) return;
  const int c = (int)(t - v * lanes) * VEC;
  F zero;
#pragma unroll
  for (int k = 0; k < VEC; ++k) zero.x[k] = 0.f;
  const int own = point2voxel_map[v];
  if (!inVoxel(own, voxel_num, rows)) {
    *reinterpret_cast<F *>(grad_feats + (size_t)v * num_features + c) = zero;
  } else if (const uint32_t place = starts[own]; (place & kUnlisted) != 0) {
    const F mine = *reinterpret_cast<const F *>(feats + (size_t)v * num_features + c);
    const F top = *reinterpret_cast<const F *>(voxel_feats + (size_t)own * num_features + c);
    int32_t *const best = from + (size_t)(place & ~kUnlisted) * num_features + c;
#pragma unroll
    for (int k = 0; k < VEC; ++k)
      if (mine.x[k] == top.x[k]) atomicMin(best + k, (int32_t)v);
  }
  if (v >= (uint32_t)min(*voxel_num, rows)) return;
  const uint32_t count = counts[v];
  if (count == 0 || count > kListed) return;
  const uint32_t begin = starts[v], stop = begin + count;
  const F top = *reinterpret_cast<const F *>(voxel_feats + (size_t)v * num_features + c);
  const F g = *reinterpret_cast<const F *>(grad_voxel_feats + (size_t)v * num_features + c);
  uint32_t best[VEC];
#pragma unroll
  for (int k = 0; k < VEC; ++k) best[k] = (uint32_t)n;
  for (uint32_t p = begin; p < stop; p += kHeld) {
    uint32_t x[kHeld];
    F mine[kHeld];
#pragma unroll
    for (int u = 0; u < kHeld; ++u) x[u] = points[min(p + u, stop - 1)];
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
      mine[u] = *reinterpret_cast<const F *>(feats + (size_t)x[u] * num_features + c);
    // (the last point of the list may be looked at again)
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
#pragma unroll
      for (int k = 0; k < VEC; ++k)
        if (mine[u].x[k] == top.x[k]) best[k] = min(best[k], x[u]);
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
      if (p + u < stop) {
        F out = zero;
        if (count <= kHeld) {
#pragma unroll
          for (int k = 0; k < VEC; ++k) out.x[k] = best[k] == x[u] ? g.x[k] : 0.f;
        }
        *reinterpret_cast<F *>(grad_feats + (size_t)x[u] * num_features + c) = out;
      }
  }
  if (count > kHeld) {
#pragma unroll
    for (int k = 0; k < VEC; ++k)
      if (best[k] < (uint32_t)n) grad_feats[(size_t)best[k] * num_features + c + k] = g.x[k];
  }
}

// The rows of the points of voxels without a list.
template <int VEC>
__global__ __launch_bounds__(kBlock) void dpvBackwardUnlisted(
    const float *__restrict__ grad_voxel_feats, const int32_t *__restrict__ point2voxel_map,
    const int32_t *__restrict__ voxel_num, int n, int num_features, int rows, const uint32_t *__restrict__ starts,
    const ListTotals *__restrict__ totals, const int32_t *__restrict__ from, float *__restrict__ grad_feats) {
  typedef Floats<VEC> F;
  if (totals->unlisted == 0) return;
  const uint32_t lanes = (uint32_t)num_features / VEC, all = (uint32_t)n * lanes;
  for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < all; t += gridDim.x * kBlock) {
    const uint32_t x = t / lanes;
    const int c = (int)(t - x * lanes) * VEC;
    const int v = point2voxel_map[x];
    if (!inVoxel(v, voxel_num, rows)) continue;
    const uint32_t place = starts[v];
    if ((place & kUnlisted) == 0) continue;
    const int32_t *const best = from + (size_t)(place & ~kUnlisted) * num_features + c;
    const F g = *reinterpret_cast<const F *>(grad_voxel_feats + (size_t)v * num_features + c);
    F out;
#pragma unroll
    for (int k = 0; k < VEC; ++k) out.x[k] = best[k] == (int32_t)x ? g.x[k] : 0.f;
    *reinterpret_cast<F *>(grad_feats + (size_t)x * num_features + c) = out;
  }
}

// ---- the same without lists ----

__global__ __launch_bounds__(kBlock) void dpvBackwardInit(float *grad_feats, size_t grad_words, int32_t *from,
                                                          size_t from_words, int32_t none) {
  const size_t stride = (size_t)gridDim.x * kBlock;
  const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
  for (size_t i = t; i < grad_words; i += stride) grad_feats[i] = 0.f;
  for (size_t i = t; i < from_words; i += stride) from[i] = none;
}

// from[v, c] = lowest point index whose feature equals the voxel's maximum
__global__ __launch_bounds__(kBlock) void dpvBackwardFindSource(
    const float *__restrict__ feats, const float *__restrict__ voxel_feats,
    const int32_t *__restrict__ point2voxel_map, int n, int num_features, int rows, int32_t *from) {
  const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= (size_t)n * num_features) return;
  const int x = (int)(t / num_features);
  const int c = (int)(t % num_features);
  const int v = point2voxel_map[x];
  if (v < 0 || v >= rows) return;
  if (feats[t] == voxel_feats[(size_t)v * num_features + c])
    atomicMin(&from[(size_t)v * num_features + c], x);
}

__global__ __launch_bounds__(kBlock) void dpvBackwardScatter(
    const float *__restrict__ grad_voxel_feats, const int32_t *__restrict__ from,
    const int32_t *__restrict__ voxel_num, int n, int num_features, int rows, float *grad_feats) {
  const size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
  const int voxels = min(*voxel_num, rows);
  if (t >= (size_t)voxels * num_features) return;
  const int x = from[t];
  if (x < n) grad_feats[(size_t)x * num_features + t % num_features] = grad_voxel_feats[t];
}

// Features a thread takes: as many as divide their number and as the tensors' alignment allows.
int featureLanes(int num_features, std::initializer_list<const void *> tensors) {
  uintptr_t low = 0;
  for (const void *p : tensors) low |= reinterpret_cast<uintptr_t>(p);
  if (num_features % 4 == 0 && low % 16 == 0) return 4;
  if (num_features % 2 == 0 && low % 8 == 0) return 2;
  return 1;
}

// From this many features in all and a point on the backward pass lists points.  A list costs the same
// for a point of any number of features, an atomic minimum a feature: at 400 k points lists take 65 us
// against 72 to 81 with 32 features and 94 against 164 to 190 with 64 (the larger figures with a voxel
// row for every point), and no less than the minima with 24 (60) and 16 (52 against 39); at 50 k
// points, where launches count, 26 against 14 with 32 features and 32 against 22 with 64.
constexpr int kFeaturesForLists = 32;
constexpr size_t kAllFeaturesForLists = 8000000;

struct Workspace {
  u64 *keys_a, *keys_b;
  uint32_t *points_a, *points_b, *counters;
  int32_t *first_pos, *block_max;
  device_sort::FlagRanks starts;
  size_t total;
};

Workspace carve(void *base, const ScatterShape &s) {
  const size_t n = (size_t)s.num_points;
  // Blocks start at the caller's pointer rounded up to 256 bytes (64-bit keys, packed sort
  // keys and the sort's counters need their alignment whatever the caller
  // passes); the reported size includes that slack.  A null base only measures.
  char *p = base ? reinterpret_cast<char *>(alignUp(reinterpret_cast<uintptr_t>(base))) : nullptr;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *q = p ? p + off : nullptr;
    off += alignUp(bytes);
    return q;
  };
  Workspace w;
  w.keys_a = reinterpret_cast<u64 *>(take(8 * n));
  w.keys_b = reinterpret_cast<u64 *>(take(8 * n));
  w.points_a = reinterpret_cast<uint32_t *>(take(4 * n));
  w.points_b = reinterpret_cast<uint32_t *>(take(4 * n));
  w.first_pos = reinterpret_cast<int32_t *>(take(4 * (n + 1)));
  w.block_max = reinterpret_cast<int32_t *>(take(4 * 3 * kPrepareBlocks));
  w.counters = reinterpret_cast<uint32_t *>(take(4 * device_sort::sortCounterWords(s.num_points)));
  w.starts.bits = reinterpret_cast<u64 *>(take(8 * device_sort::flagBitmapWords(s.num_points)));
  w.starts.before_word = reinterpret_cast<uint32_t *>(take(4 * device_sort::flagBitmapWords(s.num_points)));
  w.starts.tiles = reinterpret_cast<uint32_t *>(take(4 * device_sort::flagTileWords(s.num_points)));
  w.total = off + 256;
  return w;
}

int bitLength(u64 v) {
  int b = 1;
  while (b < 64 && (v >> b) != 0) ++b;
  return b;
}

}  // namespace

size_t scatterWorkspaceBytes(const ScatterShape &s) { return carve(nullptr, s).total; }

hipError_t launchScatterPoints(const LaunchCtx &lc, const ScatterShape &s, const float *feats,
                               int32_t *coors, void *workspace, size_t workspace_bytes,
                               unsigned long long *host_words, unsigned long long stamp, float *voxel_feats,
                               int32_t *voxel_coors, int32_t *point2voxel_map, int32_t *voxel_points_count,
                               int32_t *voxel_num) {
  const int n = s.num_points;
  Workspace w = carve(workspace, s);
  if (w.total > workspace_bytes) return hipErrorInvalidValue;
  const int blocks = gridFor((size_t)n);
  hipError_t e;

  for (int axis = 0; axis < 3; ++axis) __atomic_store_n(host_words + axis, ~stamp << 32, __ATOMIC_RELAXED);
  const int prepare_blocks = gridFor((size_t)n, kPrepareBlocks);
  lc.begin("dpvPrepare");
  dpvPrepare<<<prepare_blocks, kBlock, 0, lc.stream>>>(coors, n, w.block_max);
  dpvAxisMax<<<1, 192, 0, lc.stream>>>(w.block_max, prepare_blocks, host_words, stamp);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;
  int32_t top[3];
  for (int axis = 0; axis < 3; ++axis)
    if ((e = waitForWord(lc.stream, host_words + axis, stamp, top + axis)) != hipSuccess) return e;

  // values an axis has, the -1 of masked rows included
  const u64 d0 = (u64)((int64_t)top[0] + 2), d1 = (u64)((int64_t)top[1] + 2), d2 = (u64)((int64_t)top[2] + 2);
  const bool narrow = d1 * d2 <= 0x100000000ull && d0 * (d1 * d2) <= 0x100000000ull;
  const int bits[3] = {bitLength(d0 - 1), bitLength(d1 - 1), bitLength(d2 - 1)};
  const int total_bits = bits[0] + bits[1] + bits[2];
  TripleRadix radix = {(uint32_t)d1, (uint32_t)d2};
  SortedPoints sorted = {nullptr, nullptr};
  bool in_b = false;  // which pair of arrays a sort left its result in
  if (narrow) {
    const int key_bits = bitLength(d0 * d1 * d2 - 1);
    const int pass_bits = device_sort::sortPassBits(key_bits);
    const RecordsOfPoints first = {coors, radix, (1u << pass_bits) - 1u, w.keys_a};
    lc.begin("radixSortPairs");
    e = device_sort::partition(lc.stream, first, n, device_sort::sortDigits(pass_bits), pass_bits, w.counters);
    if (e == hipSuccess)
      e = device_sort::sortPairs<u64, false>(lc.stream, w.counters, w.keys_a, w.keys_b, nullptr, nullptr, n, pass_bits,
                                             key_bits, pass_bits, &in_b);
    lc.end();
    if (e != hipSuccess) return e;
    sorted.records = in_b ? w.keys_b : w.keys_a;
  } else if (total_bits <= 64) {
    lc.begin("dpvPackKeys");
    dpvPackKeys<<<blocks, kBlock, 0, lc.stream>>>(coors, n, bits[1], bits[2], w.keys_a, w.points_a);
    lc.end();
    if ((e = hipGetLastError()) != hipSuccess) return e;
    lc.begin("radixSortPairs");
    e = device_sort::sortPairs<u64, true>(lc.stream, w.counters, w.keys_a, w.keys_b, w.points_a, w.points_b, n, 0,
                                          total_bits, device_sort::sortPassBits(total_bits), &in_b);
    lc.end();
    if (e != hipSuccess) return e;
    sorted.points = in_b ? w.points_b : w.points_a;
  } else {
    // last axis first; every pass is stable, so the final order is lexicographic
    // with equal triples in point order
    uint32_t *points = w.points_a, *other = w.points_b;
    uint32_t *keys = reinterpret_cast<uint32_t *>(w.keys_a), *other_keys = reinterpret_cast<uint32_t *>(w.keys_b);
    for (int axis = 2; axis >= 0; --axis) {
      lc.begin("dpvAxisKeys");
      dpvAxisKeys<<<blocks, kBlock, 0, lc.stream>>>(coors, points, axis == 2, n, axis, keys);
      lc.end();
      if ((e = hipGetLastError()) != hipSuccess) return e;
      lc.begin("radixSortPairs");
      e = device_sort::sortPairs<uint32_t, true>(lc.stream, w.counters, keys, other_keys, points, other, n, 0,
                                                 bits[axis], device_sort::sortPassBits(bits[axis]), &in_b);
      lc.end();
      if (e != hipSuccess) return e;
      if (in_b) {
        uint32_t *t = points;
        points = other;
        other = t;
      }
    }
    sorted.points = points;
  }

  lc.begin("rankFlags");
  e = narrow ? device_sort::rank(lc.stream, TripleStarts<true>{sorted, coors}, n, &w.starts)
             : device_sort::rank(lc.stream, TripleStarts<false>{sorted, coors}, n, &w.starts);
  lc.end();
  if (e != hipSuccess) return e;

  lc.begin("dpvEmit");
  dpvEmit<<<blocks, kBlock, 0, lc.stream>>>(coors, sorted, radix, w.starts, n, s.voxel_rows, point2voxel_map,
                                            voxel_coors, w.first_pos, voxel_num);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (s.voxel_rows == 0) return hipSuccess;

  const int vec = featureLanes(s.num_features, {feats, voxel_feats});
  const int grid = gridFor((size_t)s.voxel_rows * (s.num_features / vec));
  auto reduce = vec == 4   ? (s.reduce_max ? dpvReduce<4, true> : dpvReduce<4, false>)
                : vec == 2 ? (s.reduce_max ? dpvReduce<2, true> : dpvReduce<2, false>)
                           : (s.reduce_max ? dpvReduce<1, true> : dpvReduce<1, false>);
  lc.begin("dpvReduce");
  reduce<<<grid, kBlock, 0, lc.stream>>>(feats, sorted, w.first_pos, voxel_num, n, s.num_features, s.voxel_rows,
                                         voxel_feats, voxel_coors, voxel_points_count);
  lc.end();
  return hipGetLastError();
}

hipError_t launchScatterPointsBackward(const LaunchCtx &lc, int num_points, int num_features,
                                       int voxel_rows, const float *grad_voxel_feats,
                                       const float *feats, const float *voxel_feats,
                                       const int32_t *point2voxel_map, const int32_t *voxel_num,
                                       void *workspace, size_t workspace_bytes, float *grad_feats) {
  const int n = num_points, rows = voxel_rows;
  hipError_t e = hipSuccess;
  // [counts, starts: a row each][points][totals][from: a row for every voxel without a list]
  const size_t unlisted_most = (size_t)n / (kListed + 1);
  const size_t list_words = 2 * (size_t)rows + n + sizeof(ListTotals) / 4 + unlisted_most * num_features;
  if (num_features >= kFeaturesForLists && (size_t)n * num_features >= kAllFeaturesForLists &&
      workspace_bytes >= 4 * list_words) {
    uint32_t *counts = static_cast<uint32_t *>(workspace), *starts = counts + rows, *points = starts + rows;
    ListTotals *totals = reinterpret_cast<ListTotals *>(points + n);
    int32_t *from = reinterpret_cast<int32_t *>(totals + 1);
    // (free words: the gradients until the last kernels)
    uint32_t *arrival = reinterpret_cast<uint32_t *>(grad_feats);
    const int list_blocks = gridFor((size_t)n);
    lc.begin("dpvBackwardLists");
    dpvBackwardClearCounts<<<gridFor((size_t)rows), kBlock, 0, lc.stream>>>(counts, rows, totals);
    dpvBackwardCount<<<(n + kCountThreads * kCountPer - 1) / (kCountThreads * kCountPer), kCountThreads, 0,
                       lc.stream>>>(point2voxel_map, voxel_num, n, rows, (uint32_t)unlisted_most, counts, arrival);
    dpvBackwardPlaces<<<rows / (kPlaceThreads * kPlacePer) + 1, kPlaceThreads, 0, lc.stream>>>(
        counts, voxel_num, rows, (uint32_t)unlisted_most, totals, starts);
    dpvBackwardList<<<list_blocks + gridFor(unlisted_most * num_features, 256), kBlock, 0, lc.stream>>>(
        point2voxel_map, voxel_num, n, rows, num_features, list_blocks, starts, arrival, points, totals, from);
    lc.end();
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const int vec = featureLanes(num_features, {feats, voxel_feats, grad_voxel_feats, grad_feats});
    const size_t threads = (size_t)n * (num_features / vec);
    auto voxels = vec == 4 ? dpvBackwardVoxels<4> : vec == 2 ? dpvBackwardVoxels<2> : dpvBackwardVoxels<1>;
    lc.begin("dpvBackwardVoxels");
    voxels<<<gridFor(threads), kBlock, 0, lc.stream>>>(grad_voxel_feats, feats, voxel_feats, point2voxel_map,
                                                       voxel_num, n, num_features, rows, counts, starts, points, from,
                                                       grad_feats);
    lc.end();
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (unlisted_most == 0) return hipSuccess;
    auto unlisted = vec == 4 ? dpvBackwardUnlisted<4> : vec == 2 ? dpvBackwardUnlisted<2> : dpvBackwardUnlisted<1>;
    lc.begin("dpvBackwardUnlisted");
    unlisted<<<gridFor(threads, 2048), kBlock, 0, lc.stream>>>(grad_voxel_feats, point2voxel_map, voxel_num, n,
                                                               num_features, rows, starts, totals, from, grad_feats);
    lc.end();
    return hipGetLastError();
  }
  int32_t *from = static_cast<int32_t *>(workspace);
  const size_t grad_words = (size_t)num_points * num_features;
  const size_t from_words = (size_t)voxel_rows * num_features;
  lc.begin("dpvBackwardInit");
  dpvBackwardInit<<<gridFor(grad_words, 4096), kBlock, 0, lc.stream>>>(grad_feats, grad_words, from,
                                                                       from_words, num_points);
  lc.end();
  e = hipGetLastError();
  if (e != hipSuccess || from_words == 0) return e;
  lc.begin("dpvBackwardFindSource");
  dpvBackwardFindSource<<<gridFor(grad_words), kBlock, 0, lc.stream>>>(
      feats, voxel_feats, point2voxel_map, num_points, num_features, voxel_rows, from);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;
  lc.begin("dpvBackwardScatter");
  dpvBackwardScatter<<<gridFor(from_words), kBlock, 0, lc.stream>>>(
      grad_voxel_feats, from, voxel_num, num_points, num_features, voxel_rows, grad_feats);
  lc.end();
  return hipGetLastError();
}

}  // namespace dynamic_point_to_voxel
}  // namespace mluop
