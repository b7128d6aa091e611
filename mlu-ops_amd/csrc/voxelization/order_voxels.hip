// Voxels in ascending order of their linear cell index.
//
// A bucket sort: the cells are cut into buckets of a power of two cells, about sixteen buckets a
// voxel, so that few voxels meet in one.  The voxels are counted by bucket, the counts
// scanned, the voxels placed into their bucket in whatever order they arrive, and each then finds
// its place inside by comparing itself with the bucket's others.  What bounds it is latency: of six
// launches, and of the atomics and comparisons where voxels cluster.  At 120 000 voxels of a scan in
// 41 x 1600 x 1408 cells: 2.7 us cleared, 9 counted, 2.5 scanned, 5.2 placed, 9.2 ranked (four buckets a
// voxel: 13.5 counted, 19.5 ranked, one key at a time); a radix sort of the 27-bit keys takes three passes
// of three launches, 18 us each.  Coordinates may lie outside the grid: their keys count as they
// are, in the first or last bucket, so the order is that of a sort by key, equal keys by voxel.
//
// Buckets can be crowded all the same: by coordinates outside the grid, by cells named often, in a grid
// of many more cells than there are buckets.  Beyond 256 voxels they are not compared one by one: the
// places are sorted in runs of 4096 first and a voxel is looked up in its bucket's runs.  us of the
// call, every voxel compared / runs (torch's keys, sort and gathers: 112 at 120 000 voxels, 330 at a million):
//   none outside the grid, 120 000 voxels       31 / 34 (the launch that finds nothing to sort)
//   a tenth outside, at one cell (spread)       2121 (1013) / 105 (101);  16 000 voxels 312 (148) / 82 (79)
//   all outside                                 22 000 (9800) / 196 (151)
//   a million voxels, a tenth (all) outside     19 400 / 318 (3600)
#include <hip/hip_runtime.h>

#include "core/wave_scan.h"
#include "voxelization/order_voxels.h"

namespace mluop {
namespace voxelization {
namespace {

constexpr int kThreads = 256;
constexpr int kTileBuckets = 4 * kThreads;  // buckets a workgroup scans
constexpr int kAtOnce = 8;                  // keys of a bucket requested together
constexpr int kMaxTiles = 1024;             // every workgroup sums their counts in LDS
constexpr int kCompared = 256;              // most voxels of a bucket that are compared with each other
constexpr int kRun = 4096;                  // places sorted together where a bucket holds more
constexpr int kRunThreads = 1024;
constexpr int kRunsAtOnce = 8;              // sorted runs searched together

struct Cells {
  const int32_t *coors;
  int64_t h, w;
  int64_t voxels;
  int shift;    // log2 of the cells of a bucket
  int buckets;  // a multiple of kTileBuckets
  __device__ int64_t key(int64_t v) const {
    const int32_t *c = coors + 3 * v;
    // (coordinates far outside the grid wrap round)
    return (int64_t)(((uint64_t)(int64_t)c[0] * (uint64_t)h + (uint64_t)(int64_t)c[1]) * (uint64_t)w +
                     (uint64_t)(int64_t)c[2]);
  }
  __device__ int bucket(int64_t key) const {
    const int64_t b = key >> shift;
    return b < 0 ? 0 : (b >= buckets ? buckets - 1 : (int)b);
  }
};

__global__ __launch_bounds__(kThreads) void orderClear(uint4 *counts, int quads, uint32_t *crowded) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < quads) counts[i] = make_uint4(0, 0, 0, 0);
  if (i == 0) *crowded = 0;
}

// Atomics on one address take 11 ns each (120 000 voxels in one bucket: 1364 us), so a workgroup's voxels
// of one bucket take their slots with one: of the threads whose buckets meet in an entry of a table in
// LDS, the one whose write stayed asks for all that are in its bucket, and the others each for
// themselves.  *crowded: some bucket holds more than kCompared voxels.
__global__ __launch_bounds__(kThreads) void orderCount(Cells cells, uint32_t *counts, uint32_t *slots,
                                                       uint32_t *crowded) {
  constexpr int kEntries = 4 * kThreads;
  __shared__ int s_who[kEntries], s_bucket[kThreads];
  __shared__ uint32_t s_together[kThreads], s_first[kThreads];
  const int tid = threadIdx.x;
  const int64_t v = (int64_t)blockIdx.x * kThreads + tid;
  const bool live = v < cells.voxels;
  const int b = live ? cells.bucket(cells.key(v)) : -1;
  if (live) s_who[b % kEntries] = tid;
  s_bucket[tid] = b;
  s_together[tid] = 0;
  __syncthreads();
  const int who = live ? s_who[b % kEntries] : tid;
  const bool joined = live && s_bucket[who] == b;
  const uint32_t mine = joined ? atomicAdd(&s_together[who], 1u) : 0u;
  __syncthreads();
  uint32_t slot = 0;
  if (live && (!joined || who == tid)) slot = atomicAdd(&counts[b], joined ? s_together[tid] : 1u);
  s_first[tid] = slot;
  __syncthreads();
  if (!live) return;
  if (joined) slot = s_first[who] + mine;
  slots[v] = slot;
  if (slot == (uint32_t)kCompared) *crowded = 1;  // (one thread of a bucket, if any)
}

// Sum of the values of the threads in front of this one; *all: of all threads.
__device__ __forceinline__ uint32_t sumInFront(uint32_t mine, uint32_t *all) {
  __shared__ uint32_t s_waves[kThreads / 64];
  const int wave = threadIdx.x >> 6;
  const uint32_t incl = (uint32_t)waveInclusiveScan((int)mine);
  if ((threadIdx.x & 63) == 63) s_waves[wave] = incl;
  __syncthreads();
  uint32_t front = 0, total = 0;
#pragma unroll
  for (int x = 0; x < kThreads / 64; ++x) {
    if (x < wave) front += s_waves[x];
    total += s_waves[x];
  }
  *all = total;
  return front + incl - mine;
}

// The counts of a tile of buckets become the voxels in front of each bucket inside its tile.
__global__ __launch_bounds__(kThreads) void orderScanTiles(uint4 *counts, uint32_t *tiles) {
  const size_t at = (size_t)blockIdx.x * kThreads + threadIdx.x;
  const uint4 c = counts[at];
  uint32_t all;
  const uint32_t front = sumInFront(c.x + c.y + c.z + c.w, &all);
  counts[at] = make_uint4(front, front + c.x, front + c.x + c.y, front + c.x + c.y + c.z);
  if (threadIdx.x == 0) tiles[blockIdx.x] = all;
}

// Voxels in front of every tile, into LDS; ends in a barrier.
__device__ __forceinline__ void sumTiles(const uint32_t *tiles, int n_tiles, uint32_t *s_front) {
  constexpr int PER = kMaxTiles / kThreads;
  uint32_t t[PER], mine = 0, all;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = threadIdx.x * PER + i;
    t[i] = at < n_tiles ? tiles[at] : 0u;
    mine += t[i];
  }
  uint32_t front = sumInFront(mine, &all);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    s_front[threadIdx.x * PER + i] = front;
    front += t[i];
  }
  __syncthreads();
}

__global__ __launch_bounds__(kThreads) void orderPlace(Cells cells, const uint32_t *starts, const uint32_t *tiles,
                                                       const uint32_t *slots, int64_t *keys, int32_t *ids) {
  __shared__ uint32_t s_front[kMaxTiles];
  sumTiles(tiles, cells.buckets / kTileBuckets, s_front);
  const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (v >= cells.voxels) return;
  const int64_t key = cells.key(v);
  const int b = cells.bucket(key);
  const uint32_t at = s_front[b / kTileBuckets] + starts[b] + slots[v];
  keys[at] = key;
  ids[at] = (int32_t)v;
}

// Where a bucket is crowded, every run of kRun places is sorted by (key, voxel).  Buckets ascend with their
// keys, so that each keeps its places.  Returns at once where none is: what a bucket costs then is
// at most kCompared comparisons a voxel.
__global__ __launch_bounds__(kRunThreads) void orderSortRuns(const uint32_t *crowded, int64_t voxels, int64_t *keys,
                                                             int32_t *ids) {
  __shared__ int64_t s_key[kRun];
  __shared__ int32_t s_id[kRun];
  if (*crowded == 0) return;
  const int64_t base = (int64_t)blockIdx.x * kRun;
  for (int i = threadIdx.x; i < kRun; i += kRunThreads) {
    const bool live = base + i < voxels;
    s_key[i] = live ? keys[base + i] : INT64_MAX;
    s_id[i] = live ? ids[base + i] : INT32_MAX;
  }
  for (int size = 2; size <= kRun; size *= 2) {
    for (int apart = size / 2; apart > 0; apart /= 2) {
      __syncthreads();
      for (int i = threadIdx.x; i < kRun / 2; i += kRunThreads) {
        const int lo = 2 * i - (i & (apart - 1)), hi = lo + apart;
        const int64_t a = s_key[lo], b = s_key[hi];
        const int32_t va = s_id[lo], vb = s_id[hi];
        const bool above = a > b || (a == b && va > vb);
        if (above == ((lo & size) == 0)) {
          s_key[lo] = b; s_key[hi] = a;
          s_id[lo] = vb; s_id[hi] = va;
        }
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kRun; i += kRunThreads) {
    if (base + i >= voxels) continue;
    keys[base + i] = s_key[i];
    ids[base + i] = s_id[i];
  }
}

// Voxels of a crowded bucket [first, end) that are in front of voxel v with this key: looked for in every
// sorted run that the bucket meets.
__device__ __forceinline__ uint32_t placeInRuns(const int64_t *keys, const int32_t *ids, uint32_t first, uint32_t end,
                                                int64_t key, int32_t v) {
  uint32_t at = 0;
  for (uint32_t run = first / kRun; run <= (end - 1) / kRun; run += kRunsAtOnce) {
    uint32_t from[kRunsAtOnce], to[kRunsAtOnce];
#pragma unroll
    for (int x = 0; x < kRunsAtOnce; ++x) {
      from[x] = (run + x) * kRun;
      to[x] = from[x] + kRun;
      from[x] = from[x] < first ? first : (from[x] < end ? from[x] : end);
      to[x] = to[x] < end ? to[x] : end;
      at -= from[x];
    }
    for (int step = kRun; step > 0; step /= 2) {  // (log2(kRun) + 1 steps)
      int64_t other[kRunsAtOnce];
      uint32_t middle[kRunsAtOnce];
#pragma unroll
      for (int x = 0; x < kRunsAtOnce; ++x) {
        middle[x] = (from[x] + to[x]) / 2;
        other[x] = keys[middle[x] < end ? middle[x] : end - 1];
      }
#pragma unroll
      for (int x = 0; x < kRunsAtOnce; ++x) {
        if (from[x] >= to[x]) continue;
        if (other[x] < key || (other[x] == key && ids[middle[x]] < v)) from[x] = middle[x] + 1;
        else to[x] = middle[x];
      }
    }
#pragma unroll
    for (int x = 0; x < kRunsAtOnce; ++x) at += from[x];
  }
  return at;
}

__global__ __launch_bounds__(kThreads) void orderRank(Cells cells, const uint32_t *starts, const uint32_t *tiles,
                                                      const int64_t *keys, const int32_t *ids, int32_t batch_index,
                                                      bool aligned, int64_t *order, int32_t *indices) {
  __shared__ uint32_t s_front[kMaxTiles];
  sumTiles(tiles, cells.buckets / kTileBuckets, s_front);
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= cells.voxels) return;
  const int64_t key = keys[i];
  const int32_t v = ids[i];
  const int b = cells.bucket(key);
  const uint32_t first = s_front[b / kTileBuckets] + starts[b];
  const uint32_t end = b + 1 < cells.buckets ? s_front[(b + 1) / kTileBuckets] + starts[b + 1] : (uint32_t)cells.voxels;
  const bool crowded = end - first > (uint32_t)kCompared;
  uint32_t at = first + (crowded ? placeInRuns(keys, ids, first, end, key, v) : 0u);
  for (uint32_t j = first; j < (crowded ? first : end); j += kAtOnce) {
    int64_t other[kAtOnce];
#pragma unroll
    for (int x = 0; x < kAtOnce; ++x) other[x] = keys[j + x < end ? j + x : end - 1];
#pragma unroll
    for (int x = 0; x < kAtOnce; ++x) {
      if (j + x >= end) break;
      at += other[x] < key;
      if (other[x] == key && j + x != i) at += ids[j + x] < v;  // (a cell named twice)
    }
  }
  order[at] = v;
  const int32_t *c = cells.coors + 3 * (int64_t)v;
  const int4 cell = make_int4(batch_index, c[0], c[1], c[2]);
  if (aligned) {
    reinterpret_cast<int4 *>(indices)[at] = cell;
  } else {
    int32_t *to = indices + 4 * (size_t)at;
    to[0] = cell.x; to[1] = cell.y; to[2] = cell.z; to[3] = cell.w;
  }
}

// Sixteen buckets a voxel, never more than the workgroups' tables of tiles hold.
void cutCells(const OrderShape &s, int *shift, int *buckets) {
  const int64_t cells = s.space[0] * s.space[1] * s.space[2];
  int64_t most = 16 * s.voxels;
  if (most < kTileBuckets) most = kTileBuckets;
  if (most > (int64_t)kMaxTiles * kTileBuckets) most = (int64_t)kMaxTiles * kTileBuckets;
  *shift = 0;
  while (((cells - 1) >> *shift) + 1 > most) ++*shift;
  const int64_t n = ((cells - 1) >> *shift) + 1;
  *buckets = (int)((n + kTileBuckets - 1) / kTileBuckets * kTileBuckets);
}

struct OrderWorkspace {
  int64_t *keys;
  uint32_t *counts, *tiles, *slots, *crowded;
  int32_t *ids;
  size_t bytes;
};

OrderWorkspace carve(const OrderShape &s, int buckets, void *base) {
  size_t at = 0;
  auto take = [&](size_t bytes) {
    char *p = static_cast<char *>(base) + at;
    at += (bytes + 255) & ~(size_t)255;
    return p;
  };
  OrderWorkspace w;
  w.keys = reinterpret_cast<int64_t *>(take((size_t)s.voxels * 8));
  w.counts = reinterpret_cast<uint32_t *>(take((size_t)buckets * 4));
  w.tiles = reinterpret_cast<uint32_t *>(take(kMaxTiles * 4));
  w.slots = reinterpret_cast<uint32_t *>(take((size_t)s.voxels * 4));
  w.ids = reinterpret_cast<int32_t *>(take((size_t)s.voxels * 4));
  w.crowded = reinterpret_cast<uint32_t *>(take(4));
  w.bytes = at + 256;  // (the base is aligned up)
  return w;
}

}  // namespace

size_t orderVoxelsWorkspaceBytes(const OrderShape &s) {
  int shift, buckets;
  cutCells(s, &shift, &buckets);
  return carve(s, buckets, nullptr).bytes;
}

hipError_t launchOrderVoxels(const LaunchCtx &lc, const OrderShape &s, const int32_t *coors, void *workspace,
                             int64_t *order, int32_t *indices) {
  Cells cells = {coors, s.space[1], s.space[2], s.voxels, 0, 0};
  cutCells(s, &cells.shift, &cells.buckets);
  const OrderWorkspace ws = carve(
      s, cells.buckets, reinterpret_cast<void *>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~(uintptr_t)255));
  const int groups = (int)((s.voxels + kThreads - 1) / kThreads), tiles = cells.buckets / kTileBuckets;
  uint4 *quads = reinterpret_cast<uint4 *>(ws.counts);
  lc.begin("orderClear");
  orderClear<<<tiles, kThreads, 0, lc.stream>>>(quads, cells.buckets / 4, ws.crowded);
  lc.end();
  lc.begin("orderCount");
  orderCount<<<groups, kThreads, 0, lc.stream>>>(cells, ws.counts, ws.slots, ws.crowded);
  lc.end();
  lc.begin("orderScanTiles");
  orderScanTiles<<<tiles, kThreads, 0, lc.stream>>>(quads, ws.tiles);
  lc.end();
  lc.begin("orderPlace");
  orderPlace<<<groups, kThreads, 0, lc.stream>>>(cells, ws.counts, ws.tiles, ws.slots, ws.keys, ws.ids);
  lc.end();
  lc.begin("orderSortRuns");
  const int runs = (int)((s.voxels + kRun - 1) / kRun);
  orderSortRuns<<<runs, kRunThreads, 0, lc.stream>>>(ws.crowded, s.voxels, ws.keys, ws.ids);
  lc.end();
  const bool aligned = (reinterpret_cast<uintptr_t>(indices) & 15) == 0;
  lc.begin("orderRank");
  orderRank<<<groups, kThreads, 0, lc.stream>>>(cells, ws.counts, ws.tiles, ws.keys, ws.ids, s.batch_index, aligned,
                                                order, indices);
  lc.end();
  return hipGetLastError();
}

}  // namespace voxelization
}  // namespace mluop
