// Stable partition by a digit of the items' keys, radix sorts made of it, and ranks among flagged
// items, for the operators that group points by cell (voxelization, dynamic point-to-voxel
// scatter).  Included by their .hip files; every function enqueues kernels only: no memset, no
// copy, no wait, no allocation, so a caller may capture the launches into a HIP graph.
//
// A partition by up to 2048 digits takes three launches:
//   countTiles     a workgroup counts the digits of its tile of items into hist[tile][digit];
//   scanColumns    the counters become exclusive prefix sums down the tiles, the digits' sums totals[];
//   partitionTiles the same tiles again: a wave owns 256 consecutive items, takes them 64 at a time in
//                  order, and an item's place among the items of its digit is (items of lower digits) +
//                  (of the digit in earlier tiles) + (in earlier waves of the tile) + (in earlier chunks
//                  of the wave) + (in lower lanes of the chunk), which keeps equal digits in their
//                  input order.
// In partitionTiles, lanes that hold the same digit find each other with a ballot per digit bit, so
// a digit that nearly every item has costs what a rare one costs; the only atomics are the
// count's integer adds in LDS.
//
// A least-significant-digit sort takes as few passes of up to 10 bits as cover the key: at 0.4 M
// records of 28 bits three passes of 10 take 33 us, four of 8 bits took 55 (each launch starts
// cold, and the counters of 1024 digits stay below the size of the records).
#ifndef MLUOP_AMD_CORE_DEVICE_SORT_H_
#define MLUOP_AMD_CORE_DEVICE_SORT_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace mluop {
namespace device_sort {

typedef unsigned long long u64;

constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kWaveChunks = 4;                          // chunks of 64 items a wave takes in a row
constexpr int kRound = kTileThreads * kWaveChunks;      // items of a tile's round
constexpr int kMaxDigits = 2048;
constexpr int kMaxTiles = 1024;
constexpr uint32_t kNoDigit = 0xffffffffu;              // an item that goes nowhere
constexpr int kSortBits = 10;                           // most bits of a sort's pass
constexpr int kFlagThreads = 256;
constexpr int kFlagTile = 4096;                         // items of a tile of flags

// A tile takes `rounds` rounds of items one after the other, so that there are at most kMaxTiles
// rows of counters.
inline int roundsFor(int64_t n) {
  const int64_t all = (n + kRound - 1) / kRound;
  return all <= kMaxTiles ? 1 : (int)((all + kMaxTiles - 1) / kMaxTiles);
}

inline int tilesFor(int64_t n) {
  const int64_t tile = (int64_t)kRound * roundsFor(n);
  return (int)((n + tile - 1) / tile);
}

// Words of counters for n items in `digits` digits: totals, then hist.
inline size_t counterWords(int64_t n, int digits) { return kMaxDigits + (size_t)tilesFor(n) * digits; }

__device__ __forceinline__ uint32_t waveInclusiveSum(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t up = __shfl_up(v, d, 64);
    if (lane >= d) v += up;
  }
  return v;
}

// hist[0..tiles)[digit] -> exclusive prefix sums down the column, its sum to totals[digit].  A
// workgroup takes 32 columns (128-byte rows), 32 groups of threads share the tiles.
constexpr int kColumns = 32;
constexpr int kColumnGroups = 32;
static __global__ __launch_bounds__(kColumns *kColumnGroups) void scanColumns(uint32_t *__restrict__ hist, int tiles,
                                                                              int digits,
                                                                              uint32_t *__restrict__ totals) {
  constexpr int kPer = kMaxTiles / kColumnGroups;
  __shared__ uint32_t s_sum[kColumnGroups][kColumns];
  const int c = threadIdx.x % kColumns, g = threadIdx.x / kColumns;
  const int per = (tiles + kColumnGroups - 1) / kColumnGroups;  // at most kPer
  const int t0 = g * per, t1 = t0 + per < tiles ? t0 + per : tiles;
  uint32_t *column = hist + blockIdx.x * kColumns + c;
  uint32_t v[kPer];
  uint32_t sum = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    // (loads at a clamped place in front of any test: conditional ones would wait for each other)
    const uint32_t there = column[(size_t)(t0 + u < tiles ? t0 + u : tiles - 1) * digits];
    v[u] = t0 + u < t1 ? there : 0u;
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) sum += v[u];
  s_sum[g][c] = sum;
  __syncthreads();
  uint32_t run = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kColumnGroups; ++w) {
    const uint32_t s = s_sum[w][c];
    run += w < g ? s : 0u;
    total += s;
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (t0 + u < t1) column[(size_t)(t0 + u) * digits] = run;
    run += v[u];
  }
  if (g == 0) totals[blockIdx.x * kColumns + c] = total;
}

// Exclusive prefix sums of totals[0..digits) into s_first, by a workgroup of kTileThreads.
__device__ inline void digitStarts(const uint32_t *__restrict__ totals, int digits, uint32_t *s_first,
                                   uint32_t *s_wave) {
  constexpr int kPer = kMaxDigits / kTileThreads;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t v[kPer], sum = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int d = tid * kPer + u;
    const uint32_t there = totals[d < digits ? d : 0];
    v[u] = d < digits ? there : 0u;
    sum += v[u];
  }
  const uint32_t incl = waveInclusiveSum(sum);
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint32_t run = incl - sum;
  for (int w = 0; w < wave; ++w) run += s_wave[w];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (tid * kPer + u < digits) s_first[tid * kPer + u] = run;
    run += v[u];
  }
}

// What is partitioned is described by an ITEMS:
//   Item load(i)         item i of the input
//   uint32_t digit(item) its digit, or kNoDigit
//   void store(to, item, i)
template <typename ITEMS>
__global__ __launch_bounds__(kTileThreads) void countTiles(ITEMS items, int64_t n, int digits, int rounds,
                                                           uint32_t *__restrict__ hist) {
  __shared__ uint32_t s_count[kMaxDigits];
  for (int d = threadIdx.x; d < digits; d += kTileThreads) s_count[d] = 0;
  __syncthreads();
  const int64_t begin = (int64_t)blockIdx.x * rounds * kRound;
  for (int round = 0; round < rounds; ++round) {
    typename ITEMS::Item item[kWaveChunks];
    const int64_t base = begin + (int64_t)round * kRound + threadIdx.x;
#pragma unroll
    for (int j = 0; j < kWaveChunks; ++j) {
      const int64_t i = base + j * kTileThreads;
      item[j] = items.load(i < n ? i : n - 1);
    }
    // (integer adds in LDS: the order they land in does not matter for a count)
#pragma unroll
    for (int j = 0; j < kWaveChunks; ++j)
      if (base + j * kTileThreads < n) {
        const uint32_t digit = items.digit(item[j]);
        if (digit != kNoDigit) atomicAdd(&s_count[digit], 1u);
      }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < digits; d += kTileThreads) hist[(size_t)blockIdx.x * digits + d] = s_count[d];
}

// (`starts`, where not null, receives the first place of every digit)
template <typename ITEMS>
__global__ __launch_bounds__(kTileThreads) void partitionTiles(ITEMS items, int64_t n, int digits, int digit_bits,
                                                               int rounds, const uint32_t *__restrict__ hist,
                                                               const uint32_t *__restrict__ totals,
                                                               uint32_t *__restrict__ starts) {
  __shared__ uint16_t s_count[kTileWaves][kMaxDigits];  // items of a digit per wave, then in the waves before
  __shared__ uint32_t s_first[kMaxDigits];              // where the next item of a digit goes
  __shared__ uint32_t s_wave[kTileWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  digitStarts(totals, digits, s_first, s_wave);
  __syncthreads();
  if (starts != nullptr && blockIdx.x == 0)
    for (int d = tid; d < digits; d += kTileThreads) starts[d] = s_first[d];
  for (int d = tid; d < digits; d += kTileThreads) s_first[d] += hist[(size_t)blockIdx.x * digits + d];
  volatile uint16_t *mine = s_count[wave];
  const u64 below = (1ull << lane) - 1ull;
  for (int round = 0; round < rounds; ++round) {
    for (int d = tid; d < digits; d += kTileThreads)
#pragma unroll
      for (int w = 0; w < kTileWaves; ++w) s_count[w][d] = 0;
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * rounds + round) * kRound + (int64_t)wave * (64 * kWaveChunks) + lane;
    typename ITEMS::Item item[kWaveChunks];
    uint32_t digit[kWaveChunks], place[kWaveChunks];
#pragma unroll
    for (int j = 0; j < kWaveChunks; ++j) item[j] = items.load(base + j * 64 < n ? base + j * 64 : n - 1);
#pragma unroll
    for (int j = 0; j < kWaveChunks; ++j) {
      digit[j] = base + j * 64 < n ? items.digit(item[j]) : kNoDigit;
      const bool valid = digit[j] != kNoDigit;
      u64 peers = __ballot(valid);
      for (int b = 0; b < digit_bits; ++b) {
        const bool bit = (digit[j] >> b) & 1u;
        const u64 with = __ballot(bit);
        peers &= bit ? with : ~with;
      }
      const int leader = valid ? __ffsll((long long)peers) - 1 : lane;
      uint32_t before = 0;  // items of the digit in the wave's earlier chunks
      if (valid && lane == leader) {
        before = mine[digit[j]];
        mine[digit[j]] = (uint16_t)(before + (uint32_t)__popcll(peers));
      }
      before = __shfl(before, leader, 64);
      place[j] = before + (uint32_t)__popcll(peers & below);
    }
    __syncthreads();
    // the waves' counts of a digit become the counts of the waves before
    uint32_t round_total[kMaxDigits / kTileThreads];
#pragma unroll
    for (int u = 0; u < kMaxDigits / kTileThreads; ++u) {
      const int d = tid + u * kTileThreads;
      uint32_t run = 0;
      if (d < digits) {
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) {
          const uint32_t c = s_count[w][d];
          s_count[w][d] = (uint16_t)run;
          run += c;
        }
      }
      round_total[u] = run;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kWaveChunks; ++j)
      if (digit[j] != kNoDigit)
        items.store((size_t)s_first[digit[j]] + s_count[wave][digit[j]] + place[j], item[j], base + j * 64);
    if (round + 1 == rounds) break;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMaxDigits / kTileThreads; ++u) {
      const int d = tid + u * kTileThreads;
      if (d < digits) s_first[d] += round_total[u];
    }
  }
}

template <typename ITEMS>
hipError_t partition(hipStream_t stream, const ITEMS &items, int64_t n, int digits, int digit_bits,
                     uint32_t *counters) {
  const int tiles = tilesFor(n), rounds = roundsFor(n);
  uint32_t *totals = counters, *hist = counters + kMaxDigits;
  countTiles<ITEMS><<<tiles, kTileThreads, 0, stream>>>(items, n, digits, rounds, hist);
  scanColumns<<<digits / kColumns, kColumns * kColumnGroups, 0, stream>>>(hist, tiles, digits, totals);
  partitionTiles<ITEMS><<<tiles, kTileThreads, 0, stream>>>(items, n, digits, digit_bits, rounds, hist, totals,
                                                            nullptr);
  return hipGetLastError();
}

// Keys, with a 32-bit value each (VALUES) or alone; a caller whose value fits beside its key in 64
// bits sorts the packed words as keys and halves the scattered stores.
template <typename K, bool VALUES>
struct KeysAndValues {
  struct Item {
    K key;
    uint32_t value;
  };
  const K *keys_in;
  const uint32_t *values_in;
  K *keys_out;
  uint32_t *values_out;
  int shift;
  uint32_t mask;
  __device__ Item load(int64_t i) const { return {keys_in[i], VALUES ? values_in[i] : 0u}; }
  __device__ uint32_t digit(const Item &t) const { return (uint32_t)(t.key >> shift) & mask; }
  __device__ void store(size_t to, const Item &t, int64_t) const {
    keys_out[to] = t.key;
    if (VALUES) values_out[to] = t.value;
  }
};

// Bits of each pass of a sort over `bits` bits.
inline int sortPassBits(int bits) {
  const int passes = (bits + kSortBits - 1) / kSortBits;
  return (bits + passes - 1) / passes;
}
inline int sortDigits(int pass_bits) { return 1 << (pass_bits > 5 ? pass_bits : 5); }  // (whole groups of columns)

// Words of counters the sorts below want at n items.
inline size_t sortCounterWords(int64_t n) { return counterWords(n, 1 << kSortBits); }

// Sorts the n pairs (keys_a[i], values_a[i]) by the bits [from_bit, bits) of the key, equal keys in
// input order, in passes of pass_bits.  Both pairs of arrays are written; *in_b tells which holds
// the result (true: keys_b / values_b).
template <typename K, bool VALUES>
hipError_t sortPairs(hipStream_t stream, uint32_t *counters, K *keys_a, K *keys_b, uint32_t *values_a,
                     uint32_t *values_b, int64_t n, int from_bit, int bits, int pass_bits, bool *in_b) {
  *in_b = false;
  if (n == 0) return hipSuccess;
  for (int shift = from_bit; shift < bits; shift += pass_bits) {
    KeysAndValues<K, VALUES> items = {*in_b ? keys_b : keys_a,     *in_b ? values_b : values_a,
                                      *in_b ? keys_a : keys_b,     *in_b ? values_a : values_b,
                                      shift,                       (1u << pass_bits) - 1u};
    const hipError_t e = partition(stream, items, n, sortDigits(pass_bits), pass_bits, counters);
    if (e != hipSuccess) return e;
    *in_b = !*in_b;
  }
  return hipSuccess;
}

// ---- ranks among flagged items -------------------------------------------------------------

// Bitmap of the flagged items, the flagged items in front of each of its words inside their tile,
// and their number in each tile.
struct FlagRanks {
  u64 *bits;
  uint32_t *before_word;
  uint32_t *tiles;  // counts; prefix sums with the sum of all behind them once `scanned`
  int tile_count;
  bool scanned;
};

// Up to kSumTiles tiles every workgroup that asks for ranks sums up the tiles' counts itself (FlagSums),
// which takes less than a launch of its own does; more are scanned before.
constexpr int kSumTiles = 1024;
inline int flagTiles(int64_t n) { return (int)((n + kFlagTile - 1) / kFlagTile); }
inline size_t flagBitmapWords(int64_t n) { return (size_t)flagTiles(n) * (kFlagTile / 64); }
inline size_t flagTileWords(int64_t n) { return (size_t)flagTiles(n) + 8; }

// FLAGS: bool flagged(i)
template <typename FLAGS>
__global__ __launch_bounds__(kFlagThreads) void rankFlags(FLAGS flags, int64_t n, FlagRanks out) {
  constexpr int kWords = kFlagTile / 64 / (kFlagThreads / 64);  // of a wave
  __shared__ u64 s_bits[kFlagTile / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = (int64_t)blockIdx.x * kFlagTile + (int64_t)wave * kWords * 64 + lane;
  bool flag[kWords];
#pragma unroll
  for (int j = 0; j < kWords; ++j) {
    const int64_t i = base + j * 64;
    flag[j] = flags.flagged(i < n ? i : n - 1) & (i < n);
  }
#pragma unroll
  for (int j = 0; j < kWords; ++j) {
    const u64 bits = __ballot(flag[j]);
    if (lane == 0) s_bits[wave * kWords + j] = bits;
  }
  __syncthreads();
  if (wave == 0) {
    const u64 bits = s_bits[lane];
    const uint32_t c = (uint32_t)__popcll(bits);
    const uint32_t incl = waveInclusiveSum(c);
    out.bits[(size_t)blockIdx.x * 64 + lane] = bits;
    out.before_word[(size_t)blockIdx.x * 64 + lane] = incl - c;
    if (lane == 63) out.tiles[blockIdx.x] = incl;
    if (lane == 0 && blockIdx.x + 1 == gridDim.x) out.tiles[gridDim.x] = 0;  // becomes the sum of all in a scan
  }
}

// data[0..m) -> exclusive prefix sums in place, by one workgroup, in rounds of 16 counters a
// thread (four 16-byte loads in flight); `data` is 16-byte aligned and has room for m rounded
// up to a multiple of four.
constexpr int kScanThreads = 1024;
constexpr int kScanPerThread = 16;
static __global__ __launch_bounds__(kScanThreads) void scanCounters(uint32_t *data, size_t m) {
  __shared__ uint32_t s_wave[kScanThreads / 64];
  __shared__ uint32_t s_round_total;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t carry = 0;
  for (size_t round0 = 0; round0 < m; round0 += (size_t)kScanThreads * kScanPerThread) {
    const size_t begin = round0 + (size_t)tid * kScanPerThread;
    uint4 q[kScanPerThread / 4];
#pragma unroll
    for (int u = 0; u < kScanPerThread / 4; ++u) {
      const size_t i = begin + 4 * u;
      q[u] = i < m ? *reinterpret_cast<const uint4 *>(data + i) : make_uint4(0, 0, 0, 0);
      // (the words of a last, partial group that lie past m count as zero)
      if (i + 1 >= m) q[u].y = 0;
      if (i + 2 >= m) q[u].z = 0;
      if (i + 3 >= m) q[u].w = 0;
    }
    uint32_t sum = 0;
#pragma unroll
    for (int u = 0; u < kScanPerThread / 4; ++u) sum += q[u].x + q[u].y + q[u].z + q[u].w;
    const uint32_t incl = waveInclusiveSum(sum);
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    if (wave == 0) {
      const uint32_t w = lane < kScanThreads / 64 ? s_wave[lane] : 0;
      const uint32_t wi = waveInclusiveSum(w);
      if (lane < kScanThreads / 64) s_wave[lane] = wi - w;
      if (lane == 63) s_round_total = wi;
    }
    __syncthreads();
    uint32_t run = carry + s_wave[wave] + incl - sum;
#pragma unroll
    for (int u = 0; u < kScanPerThread / 4; ++u) {
      const size_t i = begin + 4 * u;
      uint4 o;
      o.x = run; run += q[u].x;
      o.y = run; run += q[u].y;
      o.z = run; run += q[u].z;
      o.w = run; run += q[u].w;
      if (i < m) *reinterpret_cast<uint4 *>(data + i) = o;
    }
    carry += s_round_total;
    __syncthreads();
  }
}

// Bitmap and ranks of n items; sets ranks->tile_count and ranks->scanned.
template <typename FLAGS>
hipError_t rank(hipStream_t stream, const FLAGS &flags, int64_t n, FlagRanks *ranks) {
  ranks->tile_count = flagTiles(n);
  ranks->scanned = ranks->tile_count > kSumTiles;
  rankFlags<FLAGS><<<ranks->tile_count, kFlagThreads, 0, stream>>>(flags, n, *ranks);
  if (ranks->scanned) scanCounters<<<1, kScanThreads, 0, stream>>>(ranks->tiles, (size_t)ranks->tile_count + 1);
  return hipGetLastError();
}

// The tiles' prefix sums for a workgroup of kFlagThreads (in shared memory).
struct FlagSums {
  uint32_t tile[kSumTiles];
  uint32_t wave[kFlagThreads / 64];

  // By the whole workgroup, first; returns the number of all flagged items.
  __device__ uint32_t add(const FlagRanks &r) {
    if (r.scanned) return r.tiles[r.tile_count];
    constexpr int kPer = kSumTiles / kFlagThreads;
    const int tid = threadIdx.x, lane = tid & 63, w0 = tid >> 6;
    uint32_t v[kPer], sum = 0, all = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int t = tid * kPer + u;
      const uint32_t there = r.tiles[t < r.tile_count ? t : 0];
      v[u] = t < r.tile_count ? there : 0u;
      sum += v[u];
    }
    const uint32_t incl = waveInclusiveSum(sum);
    if (lane == 63) wave[w0] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
#pragma unroll
    for (int w = 0; w < kFlagThreads / 64; ++w) {
      run += w < w0 ? wave[w] : 0u;
      all += wave[w];
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      tile[tid * kPer + u] = run;
      run += v[u];
    }
    __syncthreads();
    return all;
  }
  // Flagged items in front of item i.
  __device__ uint32_t before(const FlagRanks &r, uint32_t i) const {
    return (r.scanned ? r.tiles[i / kFlagTile] : tile[i / kFlagTile]) + r.before_word[i >> 6] +
           (uint32_t)__popcll(r.bits[i >> 6] & ((1ull << (i & 63)) - 1ull));
  }
  __device__ static bool flagged(const FlagRanks &r, uint32_t i) { return (r.bits[i >> 6] >> (i & 63)) & 1u; }
};

}  // namespace device_sort
}  // namespace mluop

#endif  // MLUOP_AMD_CORE_DEVICE_SORT_H_
