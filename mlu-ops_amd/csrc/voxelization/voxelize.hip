// Hard voxelization (deterministic): every point is assigned to the cell of a
// regular grid it falls in; cells are numbered in the order of their first
// point, keep their first max_points points in point order, and only the
// first max_voxels cells are kept.
//
// The reference searches, for every point, all earlier points for the same
// cell (kernels/voxelization/voxelization_kernel.mlu, KernelPoint2Voxel), then
// numbers the voxels with a single core
// (kernels/voxelization/voxelization.cpp:45-53).  Here the same result comes
// from one stable partition of the points and a table in LDS:
//   1 voxCountBuckets  the cell of every point, hashed to one of up to 2048 buckets; points per
//                      (tile, bucket).  Workgroups behind the tiles clear the outputs.
//   2 scanColumns      those counters become prefix sums down the tiles
//   3 partitionTiles   the points, packed with their cells, grouped by bucket in point order
//   4 voxRankInCells   a workgroup takes a bucket in point order: its cells go into a hash table in
//                      LDS, which gives every point its rank in its cell and its cell's first point
//   5 rankFlags        bitmap of the cells' first points with prefix sums: the voxel number of a cell
//                      is the number of first points in front of its own
//   6 voxAssign        in point order: copies points and coordinates, writes the counts
// Clouds of up to kFewPoints points take three launches instead (voxTagPoints, voxRankFew, voxAssign): every
// bucket's workgroup picks its points out of all of them, and every workgroup of the last one counts the
// first points itself.
// Integer atomics only (LDS counts and table insertion): the outputs are the same bits on
// every run.
//
// What bounds it: random access.  A cell table in device memory costs a 128-byte line each way for
// every point (58 us for 1.2 M points), a full sort by cell another 70 us in nine launches.  With the
// buckets only the partition's stores and the ranks' way back to point order are scattered, and
// every other pass streams.  One crowded cell (zero-padded clouds) is one workgroup's work: 1.3 us for
// every 512 of its points, a table lookup each.
// Measured, 1.2 M points in 2048 buckets: 75 us for the six launches (13, 7, 24, 25, 6, 11), 198 us with
// cell table and sort; 23 k points: 29 us against 72 us, where launches and latency count; 4 M points
// 182 against 552 us, 8 M 359 against 1111; 120 k points, half of them in one cell, 175 against 753.
#include <hip/hip_runtime.h>

#include "core/device_sort.h"
#include "core/wave_scan.h"

#include "voxelization/voxelize.h"

namespace mluop {
namespace voxelization {
namespace {

using device_sort::u64;

constexpr int kBlock = device_sort::kFlagThreads;

inline int gridFor(size_t n, int cap = 1 << 20) {
  size_t b = (n + kBlock - 1) / kBlock;
  if (b < 1) b = 1;
  return (int)(b > (size_t)cap ? (size_t)cap : b);
}

size_t alignUp(size_t v) { return (v + 255) & ~(size_t)255; }

// ---- partition into buckets --------------------------------------------------------------

using device_sort::kMaxDigits;
using device_sort::kNoDigit;
using device_sort::kRound;
using device_sort::kTileThreads;

// Buckets of about 500 points: a bucket is one workgroup's work, while a small cloud still gives many
// workgroups something to do.  From 1.2 million points on the buckets grow.
int bucketsFor(int64_t n) {
  int b = 64;
  while (b < kMaxDigits && (int64_t)b * 600 < n) b <<= 1;
  return b;
}

__device__ inline u64 mix64(u64 k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// Cells along one axis: the float quotient rounded half away from zero.
__device__ inline int axisCells(float lo, float hi, float size) {
  const float g = roundf((hi - lo) / size);
  return (g >= 1.f && g < 2147483648.f) ? (int)g : 0;
}

// Cell index of a coordinate, or -1 outside [0, cells) (NaN included).
__device__ inline int cellIndex(float p, float lo, float size, int cells) {
  const float f = floorf((p - lo) / size);
  if (!(f >= 0.f && f < 2147483648.f)) return -1;
  const int c = (int)f;
  return c < cells ? c : -1;
}

// The cell (z, y, x) of a point, or cz < 0 outside the grid.
struct Cell {
  int cz, cy, cx, gy, gx;
  unsigned long long cells;
};
__device__ inline Cell cellOfPoint(const float *__restrict__ p, const float *__restrict__ voxel_size,
                                   const float *__restrict__ range) {
  const float sx = voxel_size[0], sy = voxel_size[1], sz = voxel_size[2];
  const float x0 = range[0], y0 = range[1], z0 = range[2];
  const int gx = axisCells(x0, range[3], sx);
  const int gy = axisCells(y0, range[4], sy);
  const int gz = axisCells(z0, range[5], sz);
  Cell c;
  c.gx = gx;
  c.gy = gy;
  c.cells = (unsigned long long)gz * (unsigned long long)gy * gx;
  c.cx = cellIndex(p[0], x0, sx, gx);
  c.cy = c.cx < 0 ? -1 : cellIndex(p[1], y0, sy, gy);
  c.cz = c.cy < 0 ? -1 : cellIndex(p[2], z0, sz, gz);
  return c;
}

__device__ inline u64 cellKey(const Cell &c) {
  return ((u64)c.cz * (u64)c.gy + c.cy) * (u64)c.gx + c.cx;
}

// A grid of fewer than 2^32 - 1 cells (the same for every thread) has 32-bit keys; in a larger
// one the cell of a partitioned point is worked out again from the point.
__device__ inline bool smallGrid(u64 cells) { return cells < 0xffffffffull; }

__device__ inline u64 gridCells(const float *__restrict__ voxel_size, const float *__restrict__ range) {
  return (u64)axisCells(range[2], range[5], voxel_size[2]) * (u64)axisCells(range[1], range[4], voxel_size[1]) *
         (u64)axisCells(range[0], range[3], voxel_size[0]);
}

// Up to four regions of 32-bit words cleared by one launch.
constexpr int kClearRegions = 4;
struct ClearRegions {
  uint32_t *base[kClearRegions];
  size_t words[kClearRegions];
};

__device__ void clearRegions(const ClearRegions &r, int block, int blocks) {
#pragma unroll
  for (int g = 0; g < kClearRegions; ++g) {
    // words in front of the first 16-byte boundary, 16-byte stores, words behind the last
    size_t head = ((16 - (reinterpret_cast<uintptr_t>(r.base[g]) & 15)) & 15) / 4;
    head = head < r.words[g] ? head : r.words[g];
    uint32_t *body = r.base[g] + head;
    const size_t body_words = r.words[g] - head;
    const size_t quads = body_words / 4;
    uint4 *dst = reinterpret_cast<uint4 *>(body);
    for (size_t i = (size_t)block * blockDim.x + threadIdx.x; i < quads; i += (size_t)blocks * blockDim.x)
      dst[i] = make_uint4(0, 0, 0, 0);
    if (block == 0) {
      if (threadIdx.x < head) r.base[g][threadIdx.x] = 0;
      if (threadIdx.x < (body_words & 3)) body[quads * 4 + threadIdx.x] = 0;
    }
  }
}

// tagged[i] = bucket of point i (kNoDigit outside the grid) above the low half of its cell key;
// hist[tile][bucket] = points of the tile in the bucket.
__global__ __launch_bounds__(kTileThreads) void voxCountBuckets(
    const float *__restrict__ points, const float *__restrict__ voxel_size, const float *__restrict__ range,
    int64_t n, int num_features, int buckets, int rounds, int tiles, u64 *__restrict__ tagged,
    uint32_t *__restrict__ hist, ClearRegions clear) {
  __shared__ uint32_t s_count[kMaxDigits];
  if ((int)blockIdx.x >= tiles) {
    clearRegions(clear, blockIdx.x - tiles, gridDim.x - tiles);
    return;
  }
  for (int b = threadIdx.x; b < buckets; b += kTileThreads) s_count[b] = 0;
  __syncthreads();
  const int64_t begin = (int64_t)blockIdx.x * rounds * kRound;
  for (int j = 0; j < rounds * device_sort::kWaveChunks; ++j) {
    const int64_t i = begin + (int64_t)j * kTileThreads + threadIdx.x;
    if (i >= n) break;
    const Cell c = cellOfPoint(points + i * num_features, voxel_size, range);
    u64 tag = (u64)kNoDigit << 32;
    if (c.cz >= 0) {
      const u64 key = cellKey(c);
      const uint32_t bucket = (uint32_t)mix64(key) & (uint32_t)(buckets - 1);
      tag = (u64)bucket << 32 | (uint32_t)key;
      atomicAdd(&s_count[bucket], 1u);
    }
    tagged[i] = tag;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < buckets; b += kTileThreads) hist[(size_t)blockIdx.x * buckets + b] = s_count[b];
}

// The points by bucket: (point index above the low half of the cell key), points of a bucket in
// their order.
struct BucketedPoints {
  typedef u64 Item;
  const u64 *tagged;
  u64 *grouped;
  __device__ Item load(int64_t i) const { return tagged[i]; }
  __device__ uint32_t digit(Item t) const { return (uint32_t)(t >> 32); }
  __device__ void store(size_t to, Item t, int64_t i) const { grouped[to] = (u64)i << 32 | (uint32_t)t; }
};

// ---- ranks inside the cells of a bucket --------------------------------------------------

constexpr uint32_t kIsFirst = 0x80000000u;

// Cells of a bucket in LDS.  FILLS: the bucket has more points than the table has
// slots to spare, and so perhaps more cells.
template <bool FILLS, typename KEY = uint32_t>
struct LdsTable {
  KEY *keys;
  uint32_t *counts, *firsts;
  uint32_t slots;  // a power of two
  uint32_t *used;  // slots taken so far (FILLS)
  static constexpr bool kFills = FILLS;
  typedef KEY Key;
  static constexpr Key kEmpty = ~Key(0);
  __device__ static void cleared() {}
};
// The same in device memory, for buckets of more cells than the LDS table holds and, but for small buckets of few
// points, for grids whose keys need 64 bits.
struct WideTable {
  u64 *keys;
  uint32_t *counts, *firsts;
  uint32_t slots;
  typedef u64 Key;
  static constexpr Key kEmpty = ~0ull;
  uint32_t *used;
  static constexpr bool kFills = false;
  // (plain stores of empty keys, then compare-and-swap by the other waves of the workgroup)
  __device__ static void cleared() { __threadfence(); }
};

// Takes the bucket's points in order, THREADS at a time.  A wave's points of one cell are put
// in order by ballots; the waves add theirs to the cell's count one after the other.  Points of a
// cell that is full already are dropped in front of all that, so that a cell with very many points
// (padding at one coordinate) costs a table lookup a point.  False (for all threads): the bucket has
// more cells than the table takes; whoever starts again writes the same ranks again.
template <int THREADS, int SLOTS, typename TABLE>
__device__ __forceinline__ bool rankBucket(const TABLE &t, const u64 *__restrict__ entries, uint32_t count,
                           const float *__restrict__ points, const float *__restrict__ voxel_size,
                           const float *__restrict__ range, int num_features, bool small_grid, uint32_t max_points,
                           volatile uint16_t *s_owner, uint32_t *__restrict__ state, uint32_t *__restrict__ first_of,
                           uint8_t *first_flags = nullptr) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (TABLE::kFills && tid == 0) *t.used = 0;
  for (uint32_t s = tid; s < t.slots; s += THREADS) {
    t.keys[s] = TABLE::kEmpty;
    t.counts[s] = 0;
  }
  TABLE::cleared();
  __syncthreads();
  u64 next = (uint32_t)tid < count ? entries[tid] : 0;
  for (uint32_t base = 0; base < count; base += THREADS) {
    const u64 entry = next;
    const uint32_t i = base + tid;
    if (i + THREADS < count) next = entries[i + THREADS];
    bool live = i < count;
    const uint32_t idx = (uint32_t)(entry >> 32);
    uint32_t slot = 0;
    bool too_many = false;
    if (live) {
      u64 key = (uint32_t)entry;
      if (!small_grid) key = cellKey(cellOfPoint(points + (size_t)idx * num_features, voxel_size, range));
      slot = (uint32_t)(mix64(key) >> 32) & (t.slots - 1);
      // (there are more slots than points, or at least THREADS empty ones in front of every round, so
      // an empty one is always reached)
      while (true) {
        const typename TABLE::Key seen = atomicCAS(&t.keys[slot], TABLE::kEmpty, (typename TABLE::Key)key);
        if (TABLE::kFills && seen == TABLE::kEmpty) too_many = atomicAdd(t.used, 1u) + THREADS >= t.slots;
        if (seen == TABLE::kEmpty || seen == (typename TABLE::Key)key) break;
        slot = (slot + 1) & (t.slots - 1);
      }
      live = t.counts[slot] < max_points;
    }
    if constexpr (TABLE::kFills) {
      if (__syncthreads_or(too_many)) return false;
    }
    if (!__syncthreads_or(live)) continue;
    // A lane that reads its own number back is alone in its wave with the slot, or the last of its
    // group to write; the groups of all other lanes are gone through one by one.
    if (live) s_owner[slot & (SLOTS - 1)] = (uint16_t)tid;
    const bool shares = live && s_owner[slot & (SLOTS - 1)] != (uint16_t)tid;
    uint32_t rank = 0, group = 1;
    int leader = lane;
    u64 open = __ballot(shares);
    while (open != 0) {
      const uint32_t s = __shfl(slot, __ffsll((long long)open) - 1, 64);
      const bool in = live && slot == s;
      const u64 same = __ballot(in);
      if (in) {
        rank = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        group = (uint32_t)__popcll(same);
        leader = __ffsll((long long)same) - 1;
      }
      open &= ~same;
    }
    uint32_t before = 0;
    const uint32_t waves = (count - base + 63) / 64;  // that have points
    for (int w = 0; w < (int)(waves < THREADS / 64 ? waves : THREADS / 64); ++w) {
      if (wave == w && live && rank == 0) {
        before = t.counts[slot];
        t.counts[slot] = before + group;
        if (before == 0) t.firsts[slot] = idx;
      }
      __syncthreads();
    }
    rank += __shfl(before, leader, 64);
    if (live && rank > 0 && rank < max_points) {
      state[idx] = rank;
      first_of[idx] = t.firsts[slot];
    }
  }
  __syncthreads();
  for (uint32_t s = tid; s < t.slots; s += THREADS) {
    const uint32_t c = t.counts[s];
    if (c == 0) continue;
    const uint32_t first = t.firsts[s];
    state[first] = kIsFirst | (c < max_points ? c : max_points);
    if (first_flags != nullptr) first_flags[first] = 1;  // (a bit each, set by atomics, took 5 us at 23 k points)
  }
  return true;
}

// state[i] (cleared before): kIsFirst | points the cell keeps, for the first point of a cell; the
// rank in the cell for another point it keeps, whose first_of[i] is the first one; 0 otherwise.
// A bucket of any number of points is ranked in LDS as long as its cells fit there, which those of a
// crowded cell do; the table in device memory takes several times as long.
//
// The ranks of one bucket's `count` points, `entries` in point order.  `wide_at`: where the bucket's share of the
// region in device memory begins.  LONG_KEYS: the keys in LDS have room for 64 bits, which up to SLOTS / 2 points need.
template <int THREADS, int SLOTS, bool LONG_KEYS>
__device__ __forceinline__ void rankCells(const float *__restrict__ points, const float *__restrict__ voxel_size,
                                          const float *__restrict__ range, int num_features, uint32_t max_points,
                                          const u64 *__restrict__ entries, uint32_t count, size_t wide_at, u64 *wide_keys,
                                          uint32_t *wide_counts, uint32_t *wide_firsts, uint32_t *__restrict__ state,
                                          uint32_t *__restrict__ first_of, uint8_t *first_flags, bool small_grid) {
  __shared__ u64 s_long_keys[LONG_KEYS ? SLOTS : SLOTS / 2];
  __shared__ uint32_t s_counts[SLOTS], s_firsts[SLOTS];
  __shared__ uint16_t s_owner[SLOTS];
  __shared__ uint32_t s_used;
  uint32_t *const s_keys = reinterpret_cast<uint32_t *>(s_long_keys);
  if constexpr (LONG_KEYS) {
    if (!small_grid && count <= SLOTS / 2) {
      LdsTable<false, u64> t = {s_long_keys, s_counts, s_firsts, 64, nullptr};
      while (t.slots < 2 * count) t.slots <<= 1;
      rankBucket<THREADS, SLOTS>(t, entries, count, points, voxel_size, range, num_features, false, max_points, s_owner,
                                 state, first_of, first_flags);
      return;
    }
  }
  if (small_grid) {
    if (__builtin_expect(count <= SLOTS / 2, 1)) {
      LdsTable<false> t = {s_keys, s_counts, s_firsts, 64, nullptr};
      while (t.slots < 2 * count) t.slots <<= 1;
      rankBucket<THREADS, SLOTS>(t, entries, count, points, voxel_size, range, num_features, true, max_points, s_owner,
                                 state, first_of, first_flags);
      return;
    }
    const LdsTable<true> t = {s_keys, s_counts, s_firsts, SLOTS, &s_used};
    if (rankBucket<THREADS, SLOTS>(t, entries, count, points, voxel_size, range, num_features, true, max_points, s_owner,
                                   state, first_of, first_flags))
      return;
  }
  // the bucket's share of the region: the largest power of two within three slots a point
  const WideTable t = {wide_keys + wide_at, wide_counts + wide_at, wide_firsts + wide_at, 1u << (31 - __clz(3 * count)),
                       nullptr};
  rankBucket<THREADS, SLOTS>(t, entries, count, points, voxel_size, range, num_features, small_grid, max_points, s_owner,
                             state, first_of, first_flags);
}

template <int THREADS, int SLOTS>
__global__ __launch_bounds__(THREADS) void voxRankInCells(
    const float *__restrict__ points, const float *__restrict__ voxel_size, const float *__restrict__ range,
    int num_features, uint32_t max_points, const u64 *__restrict__ grouped, const uint32_t *__restrict__ bucket_start,
    const uint32_t *__restrict__ totals, u64 *wide_keys, uint32_t *wide_counts, uint32_t *wide_firsts,
    uint32_t *__restrict__ state, uint32_t *__restrict__ first_of) {
  const uint32_t count = totals[blockIdx.x];
  if (count == 0) return;
  const uint32_t start = bucket_start[blockIdx.x];
  rankCells<THREADS, SLOTS, false>(points, voxel_size, range, num_features, max_points, grouped + start, count,
                                   3 * (size_t)start, wide_keys, wide_counts, wide_firsts, state, first_of, nullptr,
                                   smallGrid(gridCells(voxel_size, range)));
}

// ---- few points ---------------------------------------------------------------------------
//
// A cloud of one sweep is a chain of launches that start cold and hold a handful of workgroups: the partition
// alone took three of them, 16 of the six launches' 29 us at 23 k points.  Here a point is tagged with its
// bucket, one byte, and every bucket's workgroup, one a CU, reads all tags (sixteen a load) and puts its own points
// in order by prefix sums.  Three launches, 3.1 + 8.6 + 5.4 us at 23 k points.  What the tags and the first points'
// flags cost grows with the points.  us of the layer's call, six launches / three: 5 k points 36.6/25.8, 12 k 38.8/28.4,
// 23 k 39.1/29.1, 40 k 40.2/32.0, 65 k 41.3/39.1, which is where the line lies.
constexpr int kFewPoints = 1 << 16;
constexpr uint32_t kFewBuckets = 255;
constexpr uint32_t kFewNone = 255;                     // the tag of a point outside the grid
constexpr int kFewThreads = 512;
constexpr int kFewTags = 16 * kFewThreads;             // tags the workgroup reads in a round
constexpr int kFewRounds = kFewPoints / kFewTags;
constexpr int kFewListed = 1024;                       // points of a bucket that are listed in LDS
constexpr uint32_t kFewSlots = 2048;                   // of the table of its cells there
static_assert(kFewRounds % 2 == 0 && kFewTags < 1 << 16, "two rounds' counts in one word");

// (multiples of whole rounds: the tags behind the last point are kFewNone)
inline size_t fewTags(int64_t n) { return ((size_t)n + kFewTags - 1) / kFewTags * kFewTags; }

// A point a thread in the first `point_blocks` workgroups; the others clear.
__global__ __launch_bounds__(kBlock) void voxTagPoints(const float *__restrict__ points,
                                                       const float *__restrict__ voxel_size,
                                                       const float *__restrict__ range, int n, int num_features,
                                                       int point_blocks, int tags_end, uint32_t *__restrict__ keys,
                                                       uint8_t *__restrict__ tags, ClearRegions clear) {
  if ((int)blockIdx.x >= point_blocks) {
    clearRegions(clear, blockIdx.x - point_blocks, gridDim.x - point_blocks);
    return;
  }
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= tags_end) return;
  uint32_t tag = kFewNone;
  if (i < n) {
    const Cell c = cellOfPoint(points + (size_t)i * num_features, voxel_size, range);
    if (c.cz >= 0) {
      const u64 key = cellKey(c);
      tag = __umulhi((uint32_t)mix64(key), kFewBuckets);
      keys[i] = (uint32_t)key;
    }
  }
  tags[i] = (uint8_t)tag;
}

// Bit 7 of every byte of `word` that is `byte`.
__device__ __forceinline__ uint32_t bytesEqual(uint32_t word, uint32_t byte) {
  const uint32_t x = word ^ (byte * 0x01010101u);
  return ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu);
}

// *cursor (cleared before): points of the buckets that have taken their places in `grouped`, in no particular order:
// those with more points than the list in LDS holds.
__global__ __launch_bounds__(kFewThreads) void voxRankFew(
    const float *__restrict__ points, const float *__restrict__ voxel_size, const float *__restrict__ range, int n,
    int num_features, uint32_t max_points, const uint32_t *__restrict__ keys, const uint8_t *__restrict__ tags,
    uint32_t *cursor, u64 *grouped, u64 *wide_keys, uint32_t *wide_counts, uint32_t *wide_firsts,
    uint32_t *__restrict__ state, uint32_t *__restrict__ first_of, uint8_t *__restrict__ first_flags) {
  constexpr int kWaves = kFewThreads / 64;
  __shared__ uint32_t s_wave[kFewRounds / 2][kWaves];
  __shared__ u64 s_list[kFewListed];
  __shared__ uint32_t s_start;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t bucket = blockIdx.x;
  const int rounds = (n + kFewTags - 1) / kFewTags;
  const bool small_grid = smallGrid(gridCells(voxel_size, range));
  uint4 t[kFewRounds];
#pragma unroll
  for (int r = 0; r < kFewRounds; ++r) {
    t[r] = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (r < rounds) t[r] = reinterpret_cast<const uint4 *>(tags)[(size_t)r * kFewThreads + tid];
  }
  uint32_t match[kFewRounds];        // bit 4 q + b: byte b of word q is one of the bucket's
  uint32_t before[kFewRounds / 2];   // two rounds a word: matches of the threads before, in the wave
#pragma unroll
  for (int r = 0; r < kFewRounds; ++r) {
    match[r] = 0;
    if (r < rounds) {
      const uint32_t words[4] = {t[r].x, t[r].y, t[r].z, t[r].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t eq = bytesEqual(words[q], bucket) >> 7;
        match[r] |= ((eq | eq >> 7 | eq >> 14 | eq >> 21) & 15u) << (4 * q);
      }
    }
    if (r % 2 == 1) {
      const uint32_t mine = (uint32_t)__popc(match[r - 1]) | (uint32_t)__popc(match[r]) << 16;
      uint32_t incl = 0;
      if (r - 1 < rounds) incl = (uint32_t)waveInclusiveScan((int)mine);
      before[r / 2] = incl - mine;
      if (lane == 63) s_wave[r / 2][wave] = incl;
    }
  }
  __syncthreads();
  uint32_t count = 0, first[kFewRounds];
#pragma unroll
  for (int r = 0; r < kFewRounds; ++r) {
    const int shift = r % 2 * 16;
    first[r] = before[r / 2] >> shift & 0xffffu;
    if (r < rounds) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        if (w == wave) first[r] += count;
        count += s_wave[r / 2][w] >> shift & 0xffffu;
      }
    }
  }
  if (count == 0) return;
  // (what is listed is ranked in LDS, also in grids whose keys need 64 bits: with a table in device memory the three kernels
  // took 76 us there at 23 k points, those of the six launches take 63, these 25)
  const bool listed = count <= (uint32_t)kFewListed;
  static_assert(kFewListed <= kFewSlots / 2, "listed points have a table in LDS");
  if (!listed) {
    if (tid == 0) s_start = atomicAdd(cursor, count);
    __syncthreads();
  }
  const uint32_t start = listed ? 0u : s_start;
#pragma unroll
  for (int r = 0; r < kFewRounds; ++r) {
    uint32_t to = first[r];
    for (uint32_t left = match[r]; left != 0; left &= left - 1) {
      const uint32_t i = (uint32_t)(r * kFewTags + tid * 16 + __ffs((int)left) - 1);
      const u64 entry = (u64)i << 32 | keys[i];
      if (listed) s_list[to++] = entry;
      else grouped[start + to++] = entry;
    }
  }
  __syncthreads();
  if (!listed) {
    rankCells<kFewThreads, kFewSlots, true>(points, voxel_size, range, num_features, max_points, grouped + start, count,
                                            3 * (size_t)start, wide_keys, wide_counts, wide_firsts, state, first_of,
                                            first_flags, small_grid);
    return;
  }
  rankCells<kFewThreads, kFewSlots, true>(points, voxel_size, range, num_features, max_points, s_list, count, 0, wide_keys,
                                          wide_counts, wide_firsts, state, first_of, first_flags, small_grid);
}

// ---- voxel numbers -----------------------------------------------------------------------

// Points a bucket has on average, above which a larger table in LDS is the better one although fewer
// workgroups share a CU (us for voxRankInCells with 2048, 4096 and 8192 slots, points strewn over all
// cells: 2.0 million points 37, 41, -; 2.4: 54, 49, -; 3.0: 68, 54, -; 4.0: 318, 74, 86; 6.0: -, 153,
// 121).  The largest takes 7168 cells, buckets of 14.6 million points; from there on more and more
// buckets go to device memory (12 million points: 330 us in LDS, 2240 us there).
constexpr int64_t kPointsForLargerTable = 1100;
constexpr int64_t kPointsForLargestTable = 2400;

struct FirstPoints {
  const uint32_t *state;
  __device__ bool flagged(int64_t i) const { return (state[i] & kIsFirst) != 0; }
};

// First points in front of a point, from a byte a point (few points): every workgroup counts all of them.
struct FewFirsts {
  const uint4 *flags;
  int pieces;  // of 16 points
};
struct FewSums {
  static constexpr int kPer = kFewPoints / 16 / kBlock;  // pieces a thread sums up
  uint32_t piece[kFewPoints / 16];
  uint32_t wave[kBlock / 64];
  __device__ static uint32_t sum(uint4 f) { return (uint32_t)(__popc(f.x) + __popc(f.y) + __popc(f.z) + __popc(f.w)); }
  __device__ uint32_t add(const FewFirsts &f) {
    const int tid = threadIdx.x;
    uint4 flags[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      flags[u] = make_uint4(0, 0, 0, 0);
      if (u * kBlock < f.pieces) flags[u] = f.flags[min(u * kBlock + tid, f.pieces - 1)];
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      piece[u * kBlock + tid] = u * kBlock + tid < f.pieces ? sum(flags[u]) : 0u;
    __syncthreads();
    const int per = (f.pieces + kBlock - 1) / kBlock, first = tid * per;
    uint32_t mine = 0, all = 0;
    for (int u = 0; u < per; ++u) mine += piece[first + u];
    const uint32_t incl = (uint32_t)waveInclusiveScan((int)mine);
    if ((tid & 63) == 63) wave[tid >> 6] = incl;
    __syncthreads();
    uint32_t run = incl - mine;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) {
      run += w < (tid >> 6) ? wave[w] : 0u;
      all += wave[w];
    }
    for (int u = 0; u < per; ++u) {
      const uint32_t c = piece[first + u];
      piece[first + u] = run;
      run += c;
    }
    __syncthreads();
    return all;
  }
  __device__ uint32_t before(const FewFirsts &f, uint32_t i) const {
    const uint4 flags = f.flags[i >> 4];
    const u64 lo = (u64)flags.y << 32 | flags.x, hi = (u64)flags.w << 32 | flags.z;
    const int bits = (int)(i & 7) * 8;
    const u64 below = (1ull << bits) - 1ull;
    const bool upper = (i & 8) != 0;
    return piece[i >> 4] + (uint32_t)__popcll((upper ? hi : lo) & below) + (upper ? (uint32_t)__popcll(lo) : 0u);
  }
};

// Point i of the cloud.
template <typename FIRSTS, typename SUMS>
__global__ __launch_bounds__(kBlock) void voxAssign(
    const float *__restrict__ points, const float *__restrict__ voxel_size, const float *__restrict__ range, int64_t n,
    int num_features, const uint32_t *__restrict__ state, const uint32_t *__restrict__ first_of,
    FIRSTS firsts, bool quads, int max_points, int max_voxels,
    float *__restrict__ voxels, int32_t *__restrict__ coors, int32_t *__restrict__ num_points_per_voxel,
    int32_t *__restrict__ voxel_num, u64 *host_voxel_num, u64 stamp) {
  __shared__ SUMS s_sums;
  const int tid = threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * kBlock + tid;
  const uint32_t st = i < n ? state[i] : 0u;
  const uint32_t all = s_sums.add(firsts);
  if (blockIdx.x == 0 && tid == 0) {
    const int32_t kept = all < (uint32_t)max_voxels ? (int32_t)all : max_voxels;
    *voxel_num = kept;
    if (host_voxel_num != nullptr)
      __hip_atomic_store(host_voxel_num, stamp << 32 | (uint32_t)kept, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (st == 0) return;
  const bool is_first = (st & kIsFirst) != 0;
  const uint32_t f = is_first ? (uint32_t)i : first_of[i];
  const uint32_t r = is_first ? 0u : st;
  const uint32_t v = s_sums.before(firsts, f);
  if (v >= (uint32_t)max_voxels) return;
  const float *src = points + (size_t)i * num_features;
  float *dst = voxels + ((size_t)v * max_points + r) * num_features;
  if (quads)
    *reinterpret_cast<float4 *>(dst) = *reinterpret_cast<const float4 *>(src);
  else
    for (int k = 0; k < num_features; ++k) dst[k] = src[k];
  if (is_first) {
    num_points_per_voxel[v] = (int32_t)(st & ~kIsFirst);
    const Cell c = cellOfPoint(src, voxel_size, range);
    coors[3 * (size_t)v] = c.cz;
    coors[3 * (size_t)v + 1] = c.cy;
    coors[3 * (size_t)v + 2] = c.cx;
  }
}

struct Workspace {
  u64 *tagged, *grouped, *wide_keys;
  uint32_t *state, *first_of, *counters, *bucket_start, *wide_counts, *wide_firsts;
  // few points: cleared with `state`, in front of which they lie
  uint8_t *first_flags;
  uint32_t *cursor;
  uint32_t *cleared;
  size_t clear_words;
  uint8_t *tags;
  device_sort::FlagRanks firsts;
  size_t total;
};

Workspace carve(void *base, const VoxelizeShape &s) {
  const size_t n = (size_t)s.num_points;
  // Blocks start at the caller's pointer rounded up to 256 bytes (64-bit words need their
  // alignment whatever the caller passes); the reported size includes that slack.  A null base
  // only measures.
  char *p = base ? reinterpret_cast<char *>(alignUp(reinterpret_cast<uintptr_t>(base))) : nullptr;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *q = p ? p + off : nullptr;
    off += alignUp(bytes);
    return q;
  };
  auto words = [&](size_t count) { return reinterpret_cast<uint32_t *>(take(4 * count)); };
  auto longs = [&](size_t count) { return reinterpret_cast<u64 *>(take(8 * count)); };
  Workspace w;
  w.tagged = longs(n);
  w.grouped = longs(n);
  const bool few = s.num_points <= kFewPoints;
  const size_t flag_words = few ? (n + 15) / 16 * 4 : 0;
  w.clear_words = flag_words + (few ? 1 : 0) + n;
  w.cleared = words(w.clear_words);
  w.first_flags = reinterpret_cast<uint8_t *>(w.cleared);
  w.state = w.cleared + flag_words;
  w.cursor = w.state + n;
  w.tags = reinterpret_cast<uint8_t *>(take(few ? fewTags(s.num_points) : 0));
  w.first_of = words(n);
  w.counters = words(device_sort::counterWords(s.num_points, bucketsFor(s.num_points)));
  w.bucket_start = words(kMaxDigits);
  w.firsts.bits = longs(device_sort::flagBitmapWords(s.num_points));
  w.firsts.before_word = words(device_sort::flagBitmapWords(s.num_points));
  w.firsts.tiles = words(device_sort::flagTileWords(s.num_points));
  w.wide_keys = longs(3 * n);
  w.wide_counts = words(3 * n);
  w.wide_firsts = words(3 * n);
  w.total = off + 256;
  if (!few) {
    // a workspace that is large enough for a cloud is so for every smaller one, also across the line above, below
    // which the tags and flags come on top (65 536 points need what 67 300 would)
    VoxelizeShape most_few = s;
    most_few.num_points = kFewPoints;
    const size_t few_total = carve(nullptr, most_few).total;
    if (w.total < few_total) w.total = few_total;
  }
  return w;
}

}  // namespace

size_t voxelizeWorkspaceBytes(const VoxelizeShape &s) { return carve(nullptr, s).total; }

hipError_t launchVoxelize(const LaunchCtx &lc, const VoxelizeShape &s, const float *points,
                          const float *voxel_size, const float *coors_range, void *workspace,
                          size_t workspace_bytes, float *voxels, int32_t *coors,
                          int32_t *num_points_per_voxel, int32_t *voxel_num, unsigned long long *host_voxel_num,
                          unsigned long long stamp) {
  const int64_t n = s.num_points;
  Workspace w = carve(workspace, s);
  if (w.total > workspace_bytes) return hipErrorInvalidValue;
  const int buckets = bucketsFor(n), rounds = device_sort::roundsFor(n), tiles = device_sort::tilesFor(n);
  uint32_t *totals = w.counters, *hist = w.counters + kMaxDigits;
  int bucket_bits = 0;
  while ((1 << bucket_bits) < buckets) ++bucket_bits;

  // outputs start from zero (reference kernels/voxelization/voxelization.cpp:283-309), and no
  // point has a place yet
  ClearRegions clear;
  clear.base[0] = reinterpret_cast<uint32_t *>(voxels);
  clear.words[0] = (size_t)s.max_voxels * s.max_points * s.num_features;
  clear.base[1] = reinterpret_cast<uint32_t *>(coors);
  clear.words[1] = (size_t)s.max_voxels * 3;
  clear.base[2] = reinterpret_cast<uint32_t *>(num_points_per_voxel);
  clear.words[2] = (size_t)s.max_voxels;
  clear.base[3] = w.cleared;
  clear.words[3] = w.clear_words;
  size_t most = 0;
  for (int g = 0; g < kClearRegions; ++g) most = clear.words[g] > most ? clear.words[g] : most;
  const size_t clear_blocks = most / (4 * kTileThreads) + 1;
  const bool quads = s.num_features == 4 &&
                     ((reinterpret_cast<uintptr_t>(points) | reinterpret_cast<uintptr_t>(voxels)) & 15) == 0;
  hipError_t e;
  if (n <= kFewPoints) {
    uint32_t *keys = reinterpret_cast<uint32_t *>(w.tagged);
    const int tags_end = (int)fewTags(n), point_blocks = gridFor((size_t)tags_end);
    lc.begin("voxTagPoints");
    voxTagPoints<<<point_blocks + (int)(clear_blocks < 1024 ? clear_blocks : 1024), kBlock, 0, lc.stream>>>(
        points, voxel_size, coors_range, (int)n, s.num_features, point_blocks, tags_end, keys, w.tags, clear);
    lc.end();
    if ((e = hipGetLastError()) != hipSuccess) return e;
    lc.begin("voxRankFew");
    voxRankFew<<<kFewBuckets, kFewThreads, 0, lc.stream>>>(
        points, voxel_size, coors_range, (int)n, s.num_features, (uint32_t)s.max_points, keys, w.tags, w.cursor, w.grouped,
        w.wide_keys, w.wide_counts, w.wide_firsts, w.state, w.first_of, w.first_flags);
    lc.end();
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const FewFirsts firsts = {reinterpret_cast<const uint4 *>(w.first_flags), (int)((n + 15) / 16)};
    lc.begin("voxAssign");
    voxAssign<FewFirsts, FewSums><<<gridFor((size_t)n), kBlock, 0, lc.stream>>>(
        points, voxel_size, coors_range, n, s.num_features, w.state, w.first_of, firsts, quads, s.max_points,
        s.max_voxels, voxels, coors, num_points_per_voxel, voxel_num, host_voxel_num, stamp);
    lc.end();
    return hipGetLastError();
  }
  lc.begin("voxCountBuckets");
  voxCountBuckets<<<tiles + (int)(clear_blocks < 1024 ? clear_blocks : 1024), kTileThreads, 0, lc.stream>>>(
      points, voxel_size, coors_range, n, s.num_features, buckets, rounds, tiles, w.tagged, hist, clear);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;

  lc.begin("scanColumns");
  device_sort::scanColumns<<<buckets / device_sort::kColumns, device_sort::kColumns * device_sort::kColumnGroups, 0,
                             lc.stream>>>(hist, tiles, buckets, totals);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;

  lc.begin("partitionTiles");
  device_sort::partitionTiles<<<tiles, kTileThreads, 0, lc.stream>>>(BucketedPoints{w.tagged, w.grouped}, n, buckets,
                                                                     bucket_bits, rounds, hist, totals,
                                                                     w.bucket_start);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;

  const int64_t per_bucket = n / buckets;
  const bool largest = per_bucket > kPointsForLargestTable;
  auto rank = largest                                ? voxRankInCells<1024, 8192>
              : per_bucket > kPointsForLargerTable ? voxRankInCells<512, 4096>
                                                   : voxRankInCells<512, 2048>;
  lc.begin("voxRankInCells");
  rank<<<buckets, largest ? 1024 : 512, 0, lc.stream>>>(points, voxel_size, coors_range, s.num_features,
                                                (uint32_t)s.max_points, w.grouped, w.bucket_start, totals, w.wide_keys,
                                                w.wide_counts, w.wide_firsts, w.state, w.first_of);
  lc.end();
  if ((e = hipGetLastError()) != hipSuccess) return e;

  lc.begin("rankFlags");
  e = device_sort::rank(lc.stream, FirstPoints{w.state}, n, &w.firsts);
  lc.end();
  if (e != hipSuccess) return e;

  lc.begin("voxAssign");
  voxAssign<device_sort::FlagRanks, device_sort::FlagSums><<<gridFor((size_t)n), kBlock, 0, lc.stream>>>(
      points, voxel_size, coors_range, n, s.num_features, w.state, w.first_of, w.firsts, quads, s.max_points,
      s.max_voxels, voxels, coors, num_points_per_voxel, voxel_num, host_voxel_num, stamp);
  lc.end();
  return hipGetLastError();
}

}  // namespace voxelization
}  // namespace mluop
