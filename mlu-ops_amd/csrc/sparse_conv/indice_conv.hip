// Indice convolution kernels for gfx950: forward, backward data, backward filter.
//
// Semantics (reference test/mlu_op_gtest/pb_gtest/src/zoo/
// indice_convolution_forward/indice_convolution_forward.cpp:86-176,
// indice_convolution_backward_data/indice_convolution_backward_data.cpp:254-343,
// indice_convolution_backward_filter/indice_convolution_backward_filter.cpp:121-178):
//   forward   out[o, :]  = sum_k sum_{(i,o) in pairs[k]} feat[i, :] . W[k]
//   bwd data  dX[i, :]   = sum_k sum_{(i,o) in pairs[k]} dY[o, :] . W[k]^T
//   bwd filt  dW[k]      = sum_{(i,o) in pairs[k]} X[i, :]^T . dY[o, :]
// with fp32 accumulation and one rounding to the tensor type at the end.
//
// Forward and backward data are the same "gather convolution": every result row
// is owned by exactly one workgroup, which walks the K offsets in order and adds
// the contribution of the (at most one) gathered row per offset.  No atomics,
// no inter-workgroup reduction, so results are reproducible run to run.  The
// owner of a row finds its gathered rows through the pair lists, cut by tile of
// result rows, where they are in order, or through a dense row map
// map[k][row] -> gathered row or -1, rebuilt from indice_pairs on every call.
//
// Kernels of the gather convolution (fp16, bf16 and fp32 alike):
//  * gatherConvMfma   up to 128 channels on both sides, in MFMA blocks of 16 pairs.  Per offset the
//    rows of a tile that have a partner are compacted, so MFMA work follows the number of
//    pairs, not K x rows.  Each wave owns a column slice of the fp32 accumulator tile in LDS.
//  * gatherConvTall   the same sums for rulebooks that are thinly filled: tiles of 128 to 512 rows by 64
//    columns, with waves that only fetch beside those that multiply.
//  * gatherConvWave   the same for results of up to 32 columns, one wavefront a tile.
//  * gatherConvDense  rulebooks whose (tile, offset) pieces are well filled: accumulators in
//    registers, all rows of a tile multiplied at every offset that has a pair there.
//    gatherConvDenseStaged  the same with rows above 64 bytes brought through LDS.
//  * gatherConvSingle result rows in one pair each: the products of one offset's pairs, stored as they are.
//  * gatherConvSimt   any channel count, LDS-tiled FMA.
// A row takes nothing from the filter of an offset at which it has no pair, in any of them, also
// where that filter is not finite.  Forward stores its sums behind a ReLU where the caller asks for it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cmath>
#include <type_traits>

#include "core/wave_scan.h"
#include "sparse_conv/indice_conv.h"

namespace mluop {
namespace sparse_conv {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned short u16;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

// A workgroup barrier for LDS traffic only: what the wave wrote to or read from LDS is done,
// loads from global memory stay in flight across it (__syncthreads() would wait for them).
__device__ __forceinline__ void ldsBarrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// 16 bytes per lane from global memory straight into LDS: lane l of the wave writes bytes
// [16 l, 16 l + 16) behind `lds_address` (the same in all lanes).  Written as the instruction
// itself: the compiler then does not know of an LDS write in flight, and does not hold every
// later LDS read of the wave back until all loads have returned; the caller waits (vmcnt)
// before anybody reads what was requested.
__device__ __forceinline__ void requestToLds(const void *global, uint32_t lds_address) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds_address), "v"(global) : "memory", "m0");
}
constexpr int kMaxInlineK = 128;

// What a lane without a row of its own loads: a row of zeros in device memory.
__device__ __attribute__((aligned(256))) unsigned char kZeroRow[512];  // never written

// Pair counts per offset, passed by value for the common small kernel volumes.
struct OffsetCounts {
  int n[kMaxInlineK];
};

__device__ __forceinline__ int offsetCount(const OffsetCounts &inl, const int32_t *dev, int k) {
  return dev != nullptr ? dev[k] : inl.n[k];
}

// ---- element types ---------------------------------------------------------

// MFMA traits: an operand fragment is 16 bytes per lane (vec8: kVec elements),
// kChunk reduction channels per fragment.
struct HalfElem {
  typedef _Float16 storage;
  typedef half8 vec8;
  static constexpr int kVec = 8, kChunk = 32;
  static __device__ __forceinline__ float load(const storage *p) { return (float)*p; }
  static __device__ __forceinline__ void store(storage *p, float v) { *p = (_Float16)v; }
  static __device__ __forceinline__ bool finite(storage v) {
    return (__builtin_bit_cast(u16, v) & 0x7c00u) != 0x7c00u;
  }
  static __device__ __forceinline__ float4v mfma(vec8 a, vec8 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

struct BFloat16Elem {
  typedef u16 storage;
  typedef bf16x8 vec8;
  static constexpr int kVec = 8, kChunk = 32;
  static __device__ __forceinline__ float load(const storage *p) {
    return __uint_as_float((uint32_t)*p << 16);
  }
  static __device__ __forceinline__ void store(storage *p, float v) {
    uint32_t u = __float_as_uint(v);
    if ((u & 0x7fffffffu) > 0x7f800000u) {  // NaN stays NaN
      *p = (u16)((u >> 16) | 0x40u);
      return;
    }
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    *p = (u16)(u >> 16);
  }
  static __device__ __forceinline__ bool finite(storage v) { return (v & 0x7f80u) != 0x7f80u; }
  static __device__ __forceinline__ float4v mfma(vec8 a, vec8 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

struct FloatElem {
  typedef float storage;
  typedef float4v vec8;  // four floats: lane (m, kq) holds reduction channels 4*kq + (0..3) of a 16-chunk
  static constexpr int kVec = 4, kChunk = 16;
  static __device__ __forceinline__ float load(const storage *p) { return *p; }
  static __device__ __forceinline__ void store(storage *p, float v) { *p = v; }
  static __device__ __forceinline__ bool finite(storage v) {
    return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
  }
  // Four 16x16x4 steps; step s pairs element s of both fragments, i.e. channel
  // 4*kq + s in MFMA reduction slot kq: a permutation of the chunk's 16 channels.
  static __device__ __forceinline__ float4v mfma(vec8 a, vec8 b, float4v c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], c, 0, 0, 0);
    return c;
  }
};

// A result's last step: negative sums become zero where the caller asked for it (a NaN stays one).  The
// ReLU behind a layer by itself reads and writes the whole result again: 11 of them took 97 of 1085 us
// of an 11-layer network's call.
__device__ __forceinline__ float activated(float v, bool relu) { return relu && v < 0.f ? 0.f : v; }

// ---- row map ---------------------------------------------------------------

// A launch that is enqueued before anyone knows whether it is needed: it runs when `word` is
// null or holds `value`, and returns at once otherwise.  The row-map kernels of a forward
// call that started on the pair lists without knowing whether they are in order carry the
// verdict word and the call's ticket here.
struct RunIf {
  const unsigned long long *word;
  unsigned long long value;
};
__device__ __forceinline__ bool notWanted(const RunIf &r) { return r.word != nullptr && *r.word != r.value; }

__global__ __launch_bounds__(256) void fillInt32(int32_t *dst, size_t n, int32_t value) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * 256;
  for (; i < n; i += stride) dst[i] = value;
}

// map[k][row - row_base] = partner row, for the first indice_num[k] pairs of every offset
// whose row lies in [row_base, row_base + n_rows): the map of one chunk of result rows.
// row_col / src_col select which pair column owns the result row (1 for
// forward, 0 for backward data).  Pairs that name a row outside their tensors are ignored.
// Every workgroup leaves the number of pairs it put into the map in accepted[its index]
// (unless accepted is null).
// A map slot holds one partner.  Rulebooks built from distinct coordinates name a
// result row once per offset at most; when coordinates repeat (or the pairs are
// made up, as in test case files) several pairs of one offset can name the same
// row, and the reference adds them all.  Plain stores keep whichever of them was
// written last; every workgroup of a gather kernel records how many slots of its
// tile it found filled, and repairLostPairs adds what the other pairs would have
// contributed when those counts fall short of the number of accepted pairs.
__global__ __launch_bounds__(256) void scatterRowMap(const int32_t *pairs, int L,
                                                     OffsetCounts inl, const int32_t *dev_counts,
                                                     int row_col, int src_col, int row_base,
                                                     int n_rows, int n_src, int32_t *map,
                                                     int32_t *accepted, RunIf run_if) {
  if (notWanted(run_if)) return;
  const int k = blockIdx.y;
  const int n = offsetCount(inl, dev_counts, k);
  const int32_t *base = pairs + (size_t)k * 2 * L;
  int mine = 0;
  for (int p = blockIdx.x * 256 + threadIdx.x; p < n; p += gridDim.x * 256) {
    const int r = base[(size_t)row_col * L + p] - row_base;
    const int s = base[(size_t)src_col * L + p];
    if ((unsigned)r < (unsigned)n_rows && (unsigned)s < (unsigned)n_src) {
      map[(size_t)k * n_rows + r] = s;
      ++mine;
    }
  }
  __shared__ int s_accepted;
  if (threadIdx.x == 0) s_accepted = 0;
  __syncthreads();
  mine = waveInclusiveScan(mine);
  if ((threadIdx.x & 63) == 63 && mine != 0) atomicAdd(&s_accepted, mine);
  __syncthreads();
  if (threadIdx.x == 0 && accepted != nullptr) accepted[blockIdx.y * gridDim.x + blockIdx.x] = s_accepted;
}

// The same on a flat grid: an offset gets the workgroups its pairs need and no
// more.  The (pairs, offset) grid above is sized by the fullest offset; at 125
// offsets of which one holds a quarter of all pairs, nine in ten of its workgroups
// exit at once and their dispatch is what the kernel costs.
struct OffsetBlocks {
  int first[kMaxInlineK];  // workgroups in front of the offset's first one
};

__global__ __launch_bounds__(256) void scatterRowMapFlat(const int32_t *pairs, int L,
                                                         OffsetCounts inl, OffsetBlocks blocks,
                                                         int K, int row_col, int src_col,
                                                         int row_base, int n_rows, int n_src,
                                                         int32_t *map, int32_t *accepted, RunIf run_if) {
  if (notWanted(run_if)) return;
  // last offset whose first workgroup is not behind this one (an offset without
  // pairs shares its prefix with the next one and is never chosen)
  int lo = 0, hi = K - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (blocks.first[mid] <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
  }
  const int k = lo;
  const int p = ((int)blockIdx.x - blocks.first[k]) * 256 + threadIdx.x;
  bool ok = false;
  if (p < inl.n[k]) {
    const int32_t *base = pairs + (size_t)k * 2 * L;
    const int r = base[(size_t)row_col * L + p] - row_base;
    const int s = base[(size_t)src_col * L + p];
    ok = (unsigned)r < (unsigned)n_rows && (unsigned)s < (unsigned)n_src;
    if (ok) map[(size_t)k * n_rows + r] = s;
  }
  const int total = __syncthreads_count(ok);
  if (threadIdx.x == 0 && accepted != nullptr) accepted[blockIdx.x] = total;
}

// ---- SIMT gather convolution -------------------------------------------------
// result[r, c] = sum_k sum_q A[map[k][r], q] * B(k, q, c),
// B(k, q, c) = W[k*sK + q*sQ + c*sC].  32 x 64 result tile per block.
template <typename E>
__global__ __launch_bounds__(256) void gatherConvSimt(const typename E::storage *A, int Q,
                                                      const typename E::storage *W, int64_t sK,
                                                      int64_t sQ, int64_t sC, const int32_t *map,
                                                      int R, int K, OffsetCounts inl,
                                                      const int32_t *dev_counts, int C,
                                                      int32_t *filled, bool relu,
                                                      typename E::storage *result) {
  constexpr int TR = 32, TC = 64, QC = 32;
  int slots = 0;  // filled map slots of this tile (first wave, uniform)
  __shared__ float As[TR][QC + 1];
  __shared__ float Bs[QC][TC];
  __shared__ int s_src[TR];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int r0 = blockIdx.x * TR, c0 = blockIdx.y * TC;
  float acc[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int k = 0; k < K; ++k) {
    if (offsetCount(inl, dev_counts, k) <= 0) continue;
    int v = -1;
    if (tid < TR && r0 + tid < R) v = map[(size_t)k * R + r0 + tid];
    if (tid < TR) s_src[tid] = v;
    if (tid < 64) slots += __popcll(__ballot(v >= 0));
    if (!__syncthreads_or(v >= 0)) continue;
    // A row without a partner takes the sums it had: zero times a filter that is not finite is a NaN.
    bool has[2];
    float before[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      has[i] = s_src[ty * 2 + i] >= 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) before[i][j] = acc[i][j];
    }
    for (int q0 = 0; q0 < Q; q0 += QC) {
#pragma unroll
      for (int i = 0; i < TR * QC / 256; ++i) {
        const int e = tid + i * 256;
        const int r = e / QC, q = e % QC;
        const int src = s_src[r];
        As[r][q] = (src >= 0 && q0 + q < Q) ? E::load(A + (size_t)src * Q + q0 + q) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < QC * TC / 256; ++i) {
        const int e = tid + i * 256;
        const int q = e / TC, c = e % TC;
        Bs[q][c] = (q0 + q < Q && c0 + c < C)
                       ? E::load(W + (size_t)k * sK + (size_t)(q0 + q) * sQ + (size_t)(c0 + c) * sC)
                       : 0.f;
      }
      __syncthreads();
#pragma unroll 8
      for (int q = 0; q < QC; ++q) {
        const float a0 = As[ty * 2][q], a1 = As[ty * 2 + 1][q];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float b = Bs[q][tx * 4 + j];
          acc[0][j] += a0 * b;
          acc[1][j] += a1 * b;
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = has[i] ? acc[i][j] : before[i][j];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = r0 + ty * 2 + i;
    if (r >= R) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = c0 + tx * 4 + j;
      if (c < C) E::store(result + (size_t)r * C + c, activated(acc[i][j], relu));
    }
  }
  if (tid == 0 && blockIdx.y == 0) filled[blockIdx.x] = slots;
}

// ---- MFMA gather convolution ---------------------------------------------------

// Channels of a filter B(k, q, c) as they are, and in fragments of the kernel instance (whose numbers
// are powers of two).  `whole`: the fragments hold nothing else.
struct FilterShape {
  int q, c;
  int chunk_bits, group_bits;  // 1 << chunk_bits fragments a column, 1 << group_bits columns of 16
  bool whole;
};

// Filter repacked into MFMA operand fragments of 16 bytes per lane (VEC elements,
// CHUNK reduction channels per fragment; 8 and 32 for the 2-byte types, 4 and 16
// for float):
// packed[(((k*(C/16) + nb)*(Q/CHUNK) + kb)*64 + lane)*VEC + e]
//   = B(k, q = kb*CHUNK + VEC*(lane/16) + e, c = nb*16 + lane%16), zero for q >= Q
// (16 reduction channels of a 2-byte type fill half a fragment) and for columns beyond the
// filter's own: a filter of q x c channels runs on the instance of the next padded size.
// Behind the fragments lie K + 1 words.  Word k holds the call's ticket (a value no earlier call
// used, so nothing has to be cleared), which word K repeats, if the filter of offset k holds an
// infinity or a NaN: a kernel that multiplies rows of zeros takes such an offset apart, since zero
// times infinity is a NaN.
template <typename E>
__device__ __forceinline__ void packFilter(const typename E::storage *W, int64_t sK, int64_t sQ, int64_t sC, int K,
                                           const FilterShape &shape, typename E::storage *packed,
                                           unsigned long long ticket, int block, int blocks) {
  constexpr int VEC = E::kVec, CHUNK = E::kChunk;
  const uint32_t total = (uint32_t)K << (shape.group_bits + shape.chunk_bits + 6);  // (below 2^24 for 4096 offsets)
  unsigned long long *const nonfinite = reinterpret_cast<unsigned long long *>(packed + (size_t)total * VEC);
  if (block == 0 && threadIdx.x == 0) nonfinite[K] = ticket;
  for (uint32_t t = block * 256 + threadIdx.x; t < total; t += blocks * 256) {
    const int lane = (int)(t & 63);
    const uint32_t fragment = t >> 6;
    const int kb = (int)(fragment & ((1u << shape.chunk_bits) - 1u));
    const int nb = (int)(fragment >> shape.chunk_bits & ((1u << shape.group_bits) - 1u));
    const int k = (int)(fragment >> (shape.chunk_bits + shape.group_bits));
    const int c = nb * 16 + (lane & 15);
    const int qb = kb * CHUNK + VEC * (lane >> 4);
    const typename E::storage *const from = W + k * sK + qb * sQ + c * sC;
    typename E::storage v[VEC];
    if (shape.whole) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = from[e * sQ];
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = qb + e < shape.q && c < shape.c ? from[e * sQ] : typename E::storage(0);
    }
    bool finite = true;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      finite = finite && E::finite(v[e]);
      packed[(size_t)t * VEC + e] = v[e];
    }
    if (!finite) nonfinite[k] = ticket;
  }
}

// Rows of `bytes` bytes copied to rows of `padded_bytes` (zeros behind), by the first `blocks`
// workgroups of a launch.
struct PadRows {
  const char *from;
  char *to;
  int bytes, padded_bytes;
  int rows;
  int blocks;
};

// Element: what the row length is a multiple of.
template <typename ELEM>
__device__ __forceinline__ void padRows(const PadRows &pad) {
  const int pieces = pad.padded_bytes / 16;
  const size_t total = (size_t)pad.rows * pieces;
  constexpr int N = 16 / (int)sizeof(ELEM);
  for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (size_t)pad.blocks * 256) {
    const size_t row = t / pieces;
    const int at = (int)(t % pieces) * 16;
    const ELEM *src = reinterpret_cast<const ELEM *>(pad.from + row * pad.bytes + at);
    ELEM v[N];
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = at + e * (int)sizeof(ELEM) < pad.bytes ? src[e] : ELEM(0);
    *reinterpret_cast<uint4 *>(pad.to + row * pad.padded_bytes + at) = *reinterpret_cast<const uint4 *>(v);
  }
}

// `elems` words set to `value` by 16-byte stores from a 16-byte boundary on.
__device__ __forceinline__ void fillWords(int32_t *words, size_t elems, int32_t value, int block, int blocks) {
  const size_t quads = elems / 4;
  int4 *dst = reinterpret_cast<int4 *>(words);
  for (size_t i = (size_t)block * 256 + threadIdx.x; i < quads; i += (size_t)blocks * 256)
    dst[i] = make_int4(value, value, value, value);
  if (block == 0 && threadIdx.x < (elems & 3)) words[quads * 4 + threadIdx.x] = value;
}

// One launch for the independent preparations of the MFMA path on a row map: the first pad.blocks
// workgroups copy the gathered rows to padded ones, the next fill_blocks set the row map to -1, the others
// repack the filter.
template <typename E>
__global__ __launch_bounds__(256) void fillMapPackFilter(PadRows pad, int32_t *map, size_t map_elems,
                                                         int fill_blocks,
                                                         const typename E::storage *W, int64_t sK,
                                                         int64_t sQ, int64_t sC, int K,
                                                         FilterShape shape,
                                                         typename E::storage *packed,
                                                         unsigned long long ticket, RunIf run_if) {
  if (notWanted(run_if)) return;
  if ((int)blockIdx.x < pad.blocks) {
    padRows<typename E::storage>(pad);
    return;
  }
  const int block = (int)blockIdx.x - pad.blocks;
  if (block < fill_blocks) {
    fillWords(map, map_elems, -1, block, fill_blocks);
    return;
  }
  packFilter<E>(W, sK, sQ, sC, K, shape, packed, ticket, block - fill_blocks,
                (int)gridDim.x - pad.blocks - fill_blocks);
}

// The same in front of gatherConvSingle: fill_blocks workgroups set the result of `elems` elements to zero, where some
// of its rows are in no pair.
template <typename E>
__global__ __launch_bounds__(256) void clearResultPackFilter(PadRows pad, typename E::storage *result, size_t elems,
                                                             int fill_blocks, const typename E::storage *W, int64_t sK,
                                                             int64_t sQ, int64_t sC, int K, FilterShape shape,
                                                             typename E::storage *packed, unsigned long long ticket) {
  if ((int)blockIdx.x < pad.blocks) {
    padRows<typename E::storage>(pad);
    return;
  }
  const int block = (int)blockIdx.x - pad.blocks;
  if (block < fill_blocks) {
    constexpr int kPerWord = 4 / (int)sizeof(typename E::storage);
    fillWords(reinterpret_cast<int32_t *>(result), elems / kPerWord, 0, block, fill_blocks);
    if (elems % kPerWord != 0 && block == 0 && threadIdx.x == 0) result[elems - 1] = typename E::storage(0);
    return;
  }
  packFilter<E>(W, sK, sQ, sC, K, shape, packed, ticket, block - fill_blocks,
                (int)gridDim.x - pad.blocks - fill_blocks);
}

// ---- where a gather kernel finds the pairs of its tile -------------------------------
//
// Either a dense row map (above), or the pair lists themselves, cut by tile.  The
// second needs the column of the pairs that names the result rows to ascend strictly
// inside every offset, which is how mluOpGetIndicePairs lists them: its input-row
// column always does (backward data), its output-row column does when the input rows
// are ordered by cell (forward).  The pairs of one offset that fall into a tile of
// result rows are then one contiguous piece of the list, and a [K, tiles + 1] table
// of cut positions replaces the [K, rows] map: nothing to clear, no slot a second pair
// could lose, a few kilobytes instead of K * rows * 4 bytes.
struct MapSource {
  static constexpr bool kSegments = false;
  const int32_t *map;
  int32_t *filled;
  RunIf run_if;
};

struct SegmentSource {
  static constexpr bool kSegments = true;
  const int32_t *pairs;               // [K, 2, L]
  const int32_t *cuts;                // [K, cut_stride]: first pair of every tile, then the count
  const unsigned long long *verdict;  // holds `ticket` when some list is not in order
  unsigned long long ticket;
  // Lists out of order: true = the kernel returns at once (row-map kernels enqueued behind
  // it do the call's work), false = every tile collects its pairs by reading all of them.
  bool leave_if_unordered;
  int L, row_col, src_col, n_src, cut_stride;
  const void *W;                      // the filter as the caller passed it, for lists out of order
  int64_t sK, sQ, sC;
  OffsetCounts counts;
};

// The pairs of one tile of result rows [r_begin, r_end) when the lists cannot be cut:
// every workgroup reads all pairs of all offsets, and each pair that names one of its
// rows is multiplied by one wave, a lane per result column, and added to the tile's
// fp32 rows in LDS (`acc`, cleared by the caller).  Offsets are taken in order with a
// barrier between them, so a row sees its offsets in the order the list kernels use;
// only rows that several pairs of one offset name depend on timing in their last
// bits.  It is slow and runs only when a pair tensor was changed
// after the library had seen it in order.
template <typename E, int NT>
__device__ __forceinline__ void scanAllPairsForTile(const typename E::storage *A, int Q, int row_bytes,
                                                    const SegmentSource &src, int K, int r_begin,
                                                    int r_end, int C, int col0, float *acc,
                                                    int acc_stride) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const typename E::storage *W = static_cast<const typename E::storage *>(src.W);
  for (int k = 0; k < K; ++k) {
    const int n = src.counts.n[k];
    const int32_t *row_list = src.pairs + ((size_t)k * 2 + src.row_col) * src.L;
    const int32_t *src_list = src.pairs + ((size_t)k * 2 + src.src_col) * src.L;
    for (int p0 = 0; p0 < n; p0 += NT) {
      const int p = p0 + tid;
      int r = -1, g = -1;
      if (p < n) {
        r = row_list[p];
        g = src_list[p];
      }
      const bool hit = r >= r_begin && r < r_end && (unsigned)g < (unsigned)src.n_src;
      unsigned long long m = __ballot(hit);
      while (m) {
        const int from = __ffsll((long long)m) - 1;
        m &= m - 1;
        const int rr = __shfl(r, from, kWave) - r_begin;
        const typename E::storage *a = reinterpret_cast<const typename E::storage *>(
            reinterpret_cast<const char *>(A) + (size_t)__shfl(g, from, kWave) * row_bytes);
        for (int c = lane; c < C; c += kWave) {
          const typename E::storage *w = W + (size_t)k * src.sK + (size_t)(col0 + c) * src.sC;
          float dot = 0.f;
          for (int q = 0; q < Q; ++q) dot += E::load(a + q) * E::load(w + (size_t)q * src.sQ);
          atomicAdd(&acc[rr * acc_stride + c], dot);
        }
      }
    }
    __syncthreads();
  }
}

// One launch in front of a gather kernel that reads pair lists: the first
// `pack_blocks` workgroups repack the filter into operand fragments (as
// fillMapPackFilter does), the others walk the pair lists, one pair per lane, and
//  * check what the gather kernel relies on: result rows in range and strictly
//    ascending inside the offset, gathered rows in range.  A violation stores `ticket`
//    in *verdict (a value no earlier call used, so the word needs no clearing);
//  * write the cut table: pair p is the first pair of every tile after its
//    predecessor's tile up to its own, and the last pair of an offset closes the
//    remaining tiles with the pair count (an offset without pairs gets one workgroup
//    that closes all its tiles with 0).  A lane with more than a few tiles to close
//    hands them to the whole wave.
constexpr int kCutPairsPerThread = 4;

template <typename E>
__global__ __launch_bounds__(256) void packFilterCutPairLists(
    PadRows pad, const typename E::storage *W, int64_t sK, int64_t sQ, int64_t sC, int K, FilterShape shape,
    typename E::storage *packed, int pack_blocks, const int32_t *pairs, int L, OffsetCounts inl,
    OffsetBlocks blocks, int row_col, int src_col, int R, int n_src, int tile_shift, int n_tiles,
    int32_t *cuts, unsigned long long *verdict, unsigned long long ticket) {
  if ((int)blockIdx.x < pad.blocks) {
    padRows<typename E::storage>(pad);
    return;
  }
  if ((int)blockIdx.x - pad.blocks < pack_blocks) {
    packFilter<E>(W, sK, sQ, sC, K, shape, packed, ticket, (int)blockIdx.x - pad.blocks, pack_blocks);
    return;
  }
  const int b = (int)blockIdx.x - pad.blocks - pack_blocks;
  int lo = 0, hi = K - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (blocks.first[mid] <= b) lo = mid; else hi = mid - 1;
  }
  const int k = lo;
  const int n = inl.n[k];
  const int lane = threadIdx.x & 63;
  const int32_t *row_list = pairs + ((size_t)k * 2 + row_col) * L;
  const int32_t *src_list = pairs + ((size_t)k * 2 + src_col) * L;
  int32_t *row_cuts = cuts + (size_t)k * (n_tiles + 1);
  // kCutPairsPerThread pairs a thread, 256 apart: all their loads are requested first
  const int p0 = (b - blocks.first[k]) * (256 * kCutPairsPerThread) + (int)threadIdx.x;
  int rs[kCutPairsPerThread], prevs[kCutPairsPerThread], ss[kCutPairsPerThread];
#pragma unroll
  for (int j = 0; j < kCutPairsPerThread; ++j) {
    const int p = p0 + j * 256;
    rs[j] = 0;
    prevs[j] = -1;
    ss[j] = 0;
    if (p < n) {
      rs[j] = row_list[p];
      ss[j] = src_list[p];
      if (p > 0) prevs[j] = row_list[p - 1];
    }
  }
#pragma unroll
  for (int j = 0; j < kCutPairsPerThread; ++j) {
    const int p = p0 + j * 256;
    const bool live = p < n;
    const int r = rs[j], prev = prevs[j], s = ss[j];
    const bool ok = (unsigned)r < (unsigned)R && (unsigned)s < (unsigned)n_src && r > prev;
    if (live && !ok) *verdict = ticket;
    // tiles (t_lo .. t_mid] open at p, tiles (t_mid .. n_tiles] close with n; clamped so
    // that a list out of order, whose table nobody reads, still writes inside the table
    int t_mid = r >> tile_shift;
    t_mid = t_mid < 0 ? 0 : (t_mid > n_tiles - 1 ? n_tiles - 1 : t_mid);
    int t_lo = p == 0 ? -1 : (prev >> tile_shift);
    t_lo = t_lo < -1 ? -1 : (t_lo > t_mid ? t_mid : t_lo);
    // job 0: value p over (t_lo, t_mid]; job 1 (last pair only): value n over (t_mid, n_tiles]
#pragma unroll
    for (int job = 0; job < 2; ++job) {
      // (an offset without pairs has one workgroup, whose first lane closes all tiles with 0)
      const bool empty_offset = n == 0 && threadIdx.x == 0 && j == 0;
      const int first = empty_offset ? 0 : (job == 0 ? t_lo + 1 : t_mid + 1);
      const int last = job == 0 ? t_mid : n_tiles;
      const int value = job == 0 ? p : n;
      const bool mine = ((live && (job == 0 || p == n - 1)) || (empty_offset && job == 1)) && first <= last;
      const bool wide = mine && last - first >= 4;
      if (mine && !wide)
        for (int t = first; t <= last; ++t) row_cuts[t] = value;
      unsigned long long m = __ballot(wide);
      while (m) {
        const int from = __ffsll((long long)m) - 1;
        m &= m - 1;
        const int f = __shfl(first, from, kWave), l = __shfl(last, from, kWave);
        const int v = __shfl(value, from, kWave);
        for (int t = f + lane; t <= l; t += kWave) row_cuts[t] = v;
      }
    }
  }
}

constexpr int mfmaTileRows(int C) {
  // fp32 accumulator tile of about 34 KiB
  return C <= 64 ? 128 : 64;
}
constexpr int mfmaColBlocksPerWave(int C) { return C >= 128 ? 2 : 1; }
// as many fetching waves as multiplying waves (five-wave workgroups place badly on the CU)
constexpr int mfmaThreads(int C) { return 128 * (C / 16 / mfmaColBlocksPerWave(C)); }
// Register budget: two eight-wave workgroups per CU need four waves per SIMD
// (128 registers a lane); the fp32 128x128 instance holds 128 registers of
// filter fragments alone and stays at one workgroup per CU.
constexpr int mfmaWavesPerSimd(int elem_bytes, int Q, int C) {
  return (elem_bytes == 4 && Q == 128 && C == 128) ? 2 : (C >= 64 ? 4 : (C == 32 ? 3 : 2));
}
constexpr int kOffsetChunk = 28;  // offsets whose pair lists are resident in LDS at once
// Gathered rows staged in LDS per round: about 25 KiB, which one wave can hold
// in registers while they travel (at most 24 16-byte pieces per lane).
constexpr int mfmaStageRows(int row_bytes) {
  return row_bytes <= 64 ? 256 : (row_bytes <= 128 ? 192 : (row_bytes <= 256 ? 96 : 48));
}
// 16-pair blocks multiplied together; bounded by the registers the W fragments of two batches
// take (16 bytes per lane for every 16-byte piece of a row and every 16 result columns).
constexpr int mfmaBatchBlocks(int elem_bytes, int Q, int C) {
  const int regs_per_block = ((Q * elem_bytes + 63) / 64) * mfmaColBlocksPerWave(C) * 4;
  const int g = 32 / regs_per_block;
  return g < 1 ? 1 : (g > 4 ? 4 : g);
}

// The rows a gather kernel reads and writes, in their own channel counts: an instance is
// compiled for padded counts, reads nothing behind a row's own bytes (a piece of 16 bytes that
// is not there is zero) and writes the result's own columns only.
struct ConvRows {
  int q;          // reduction channels
  int row_bytes;  // bytes from one gathered row to the next: a multiple of 16, all of them readable
  int c;          // result columns
  int c_padded;   // result columns of the packed filter
  bool relu;      // negative results become zero
};

// `VALS` consecutive result values of one row from column `col` on, as many as the row has.
template <typename E, int VALS>
__device__ __forceinline__ void storeColumns(typename E::storage *row, int col, int columns,
                                             const typename E::storage (&v)[VALS]) {
  typedef typename E::storage S;
  constexpr int BYTES = VALS * (int)sizeof(S);
  static_assert(BYTES == 8 || BYTES == 16, "one store");
  if (col + VALS <= columns && columns % VALS == 0) {
    if constexpr (BYTES == 8)
      *reinterpret_cast<uint2 *>(row + col) = *reinterpret_cast<const uint2 *>(v);
    else
      *reinterpret_cast<uint4 *>(row + col) = *reinterpret_cast<const uint4 *>(v);
    return;
  }
#pragma unroll
  for (int e = 0; e < VALS; ++e)
    if (col + e < columns) row[col + e] = v[e];
}

// Workgroup = TR result rows x C columns (column group blockIdx.y of the
// result's columns), WAVES multiplying waves and as many fetching waves.
// Multiplying wave w owns columns [w*16*NB, (w+1)*16*NB) of the
// fp32 accumulator tile in LDS, so no two waves ever touch the same accumulator
// element and every element sees its contributions in ascending offset order.
//
// Per chunk of kOffsetChunk offsets:
//   A   wave w (of all waves) loads map[k][row] for the offsets k = w (mod all
//       waves) of the chunk and all rows of the tile, ballots which rows have a
//       partner and, after the per-offset counts have been exchanged, compacts
//       one entry per pair (partner row << 8 | result row) into a flat list
//       ordered by offset.  The list is cut into blocks of up to 16 entries of
//       one offset, and the block list is padded to a whole batch.
//   B   the flat list is walked in rounds of STEP entries.  The partner rows of
//       a round are fetched by the fetching waves alone, with row-contiguous
//       16-byte loads (fetching them in the MFMA operand's own lane order
//       touches 16 rows per load and runs at a third of the L1 rate, once per
//       column wave), and written to the LDS stage between two barriers when
//       the multiplying waves have finished the round before.  Waves of their
//       own keep these loads out of the multiplying waves' in-order load
//       counter, where waiting for the next W fragments would also wait for
//       them.  Every multiplying wave reads its operand fragments from the
//       staged rows, multiplies W[k]^T (16 result columns x Q, fetched one
//       batch ahead) by the block's rows (Q x 16 pairs), which leaves four
//       consecutive result columns of one pair in every lane, and adds them to
//       the accumulator row of that pair with one 16-byte read-modify-write.
//       Lanes past the end of a short block repeat its first entry and
//       accumulate into a spare row.
template <typename E, int Q, int C, typename SRC>
__global__ __launch_bounds__(mfmaThreads(C))
    __attribute__((amdgpu_waves_per_eu(mfmaWavesPerSimd((int)sizeof(typename E::storage), Q, C),
                                       mfmaWavesPerSimd((int)sizeof(typename E::storage), Q, C))))
void gatherConvMfma(const typename E::storage *A, ConvRows rows, const typename E::storage *packedW,
                    SRC source, int R, int K, typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int NB = mfmaColBlocksPerWave(C);
  constexpr int WAVES = C / 16 / NB;            // multiplying waves
  constexpr int NT = mfmaThreads(C);
  constexpr int TR = mfmaTileRows(C);
  constexpr int NSEG = TR / 64;
  constexpr int KB = (Q + E::kChunk - 1) / E::kChunk;  // operand fragments per row
  constexpr bool kPartialFragment = Q < E::kChunk;     // 16 channels of a 2-byte type: upper lanes are zero
  constexpr int KC = kOffsetChunk;
  constexpr int ALLW = NT / 64;                 // multiplying + fetching waves
  constexpr int FW = ALLW - WAVES;              // fetching waves
  constexpr int KPW = (KC + ALLW - 1) / ALLW;   // offsets a wave scans per chunk
  constexpr int G = mfmaBatchBlocks((int)sizeof(S), Q, C);
  constexpr int GROUPS = C / 16;
  constexpr int MAX_ENT = KC * TR;
  constexpr int MAX_BLK = KC * (TR / 16) + G;
  constexpr int ACC_STRIDE = C + 4;             // floats; rows 16 apart fall into distinct banks
  constexpr int ROW_BYTES = Q * (int)sizeof(S);  // one gathered row
  constexpr int STAGE_STRIDE = ROW_BYTES + 16;  // padded: 16 rows x 16 bytes hit 64 distinct banks
  constexpr int PPR = ROW_BYTES / 16;           // 16-byte pieces per row
  constexpr int SROWS = mfmaStageRows(ROW_BYTES);
  constexpr int STEP = SROWS - G * 16;          // a batch starting inside a round ends inside its stage
  constexpr int PT = SROWS * PPR / (64 * FW);   // pieces per lane of a fetching wave
  static_assert(SROWS * PPR % (64 * FW) == 0 && PT <= 24, "stage must split evenly over the fetching waves");
  static_assert(KC <= 64 && MAX_ENT <= 65536 && TR <= 256, "descriptor packing");

  __shared__ __attribute__((aligned(16))) float s_acc[(TR + 1) * ACC_STRIDE];
  __shared__ __attribute__((aligned(16))) char s_stage[SROWS * STAGE_STRIDE];
  __shared__ uint32_t s_ent[MAX_ENT];   // partner row << 8 | result row in the tile
  __shared__ uint32_t s_blk[MAX_BLK];   // offset in chunk << 24 | first entry << 8 | entries
  __shared__ int s_cnt[KC];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool fetcher = wave >= WAVES;
  const int ftid = tid - 64 * WAVES;            // thread index among the fetching waves
  // Workgroups go to the eight XCDs round robin; giving XCD x the x-th eighth of the
  // tiles keeps neighbouring tiles, which gather many of the same rows, on one L2.
  const int tiles_per_xcd = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  const int r0 = tile * TR;
  if constexpr (!SRC::kSegments) {
    if (notWanted(source.run_if)) return;
  }
  if (r0 >= R) {
    if constexpr (!SRC::kSegments) {
      if (tid == 0 && blockIdx.y == 0) source.filled[blockIdx.x] = 0;
    }
    return;
  }
  int slots = 0;  // filled map slots of this tile
  const unsigned long long lt_mask = (1ull << lane) - 1ull;

  for (int i = tid; i < (TR + 1) * ACC_STRIDE; i += NT) s_acc[i] = 0.f;

  // Pair lists that turned out not to be in order (a caller who changed the tensor
  // behind the library's back): the tile collects its pairs by reading all of them.
  bool in_order = true;
  if constexpr (SRC::kSegments) {
    in_order = *source.verdict != source.ticket;
    if (!in_order && source.leave_if_unordered) return;
    if (!in_order) {
      __syncthreads();
      const int columns = rows.c - (int)blockIdx.y * C;
      scanAllPairsForTile<E, NT>(A, rows.q, rows.row_bytes, source, K, r0, r0 + TR < R ? r0 + TR : R,
                                 columns < C ? columns : C, blockIdx.y * C, s_acc, ACC_STRIDE);
    }
  }

  // per-lane constants of the multiply phase
  const char *a_bytes = reinterpret_cast<const char *>(A);
  // the workgroup owns result columns [blockIdx.y*C, (blockIdx.y+1)*C)
  const int col_group = blockIdx.y;
  const char *b_base = reinterpret_cast<const char *>(packedW) +
                       ((size_t)(col_group * GROUPS + wave * NB) * KB * 64 + lane) * 16;
  const uint32_t kBytesPerOffset = (uint32_t)(rows.c_padded / 16) * KB * 64 * 16;  // packed W[k]
  const int pair = lane & 15;
  const int quad = lane >> 4;
  char *acc_lane = reinterpret_cast<char *>(s_acc) + (wave * 16 * NB + 4 * quad) * 4;
  const char *stage_lane = s_stage + quad * 16;

  for (int kc = 0; kc < (in_order ? K : 0); kc += KC) {
    const int kn = (K - kc) < KC ? (K - kc) : KC;
    // A: the pairs of this wave's offsets; unconditional loads from clamped
    // addresses keep all of them in flight.
    int idx[KPW][NSEG];   // partner row, or -1
    int own[KPW][NSEG];   // result row inside the tile (pair lists only)
    if constexpr (SRC::kSegments) {
      // lane 2j + e fetches cut e of this wave's j-th offset
      int cut = 0;
      {
        const int kk = wave + (lane >> 1) * ALLW;
        if ((lane >> 1) < KPW && kk < kn)
          cut = source.cuts[(size_t)(kc + kk) * source.cut_stride + tile + (lane & 1)];
      }
      int first[KPW], count[KPW];
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int kk = wave + j * ALLW;
        first[j] = __shfl(cut, 2 * j, kWave);
        const int end = __shfl(cut, 2 * j + 1, kWave);
        int c = end - first[j];
        c = c < 0 ? 0 : (c > TR ? TR : c);
        count[j] = (kk < kn && source.counts.n[kk < kn ? kc + kk : kc] > 0) ? c : 0;
        const int k_safe = kk < kn ? kc + kk : kc;
        const int32_t *row_list = source.pairs + ((size_t)k_safe * 2 + source.row_col) * source.L;
        const int32_t *src_list = source.pairs + ((size_t)k_safe * 2 + source.src_col) * source.L;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          int p = first[j] + seg * 64 + lane;
          p = p < 0 ? 0 : (p < source.L ? p : source.L - 1);
          own[j][seg] = row_list[p];
          idx[j][seg] = src_list[p];
        }
      }
#pragma unroll
      for (int j = 0; j < KPW; ++j)
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) asm volatile("" : "+v"(idx[j][seg]), "+v"(own[j][seg]));
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int kk = wave + j * ALLW;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          if (seg * 64 + lane >= count[j]) idx[j][seg] = -1;
          own[j][seg] = (own[j][seg] - r0) & (TR - 1);
        }
        if (lane == 0 && kk < KC) s_cnt[kk] = count[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int kk = wave + j * ALLW;
        const int k_safe = kk < kn ? kc + kk : kc;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          const int r = r0 + seg * 64 + lane;
          idx[j][seg] = source.map[(size_t)k_safe * R + (r < R ? r : R - 1)];
          own[j][seg] = seg * 64 + lane;
        }
      }
      // Pinning the loaded values here keeps the loads above unconditional and all
      // in flight; selecting on them directly lets the compiler branch around
      // every single load and wait for it.
#pragma unroll
      for (int j = 0; j < KPW; ++j)
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) asm volatile("" : "+v"(idx[j][seg]));
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int kk = wave + j * ALLW;
        int c = 0;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          const int r = r0 + seg * 64 + lane;
          if (!(kk < kn && r < R)) idx[j][seg] = -1;
          c += __popcll(__ballot(idx[j][seg] >= 0));
        }
        if (lane == 0 && kk < KC) s_cnt[kk] = c;
      }
    }
    __syncthreads();
    // every wave scans the counts: entries and blocks in front of each offset
    const int cnt = lane < KC ? s_cnt[lane < KC ? lane : 0] : 0;
    const int nb_mine = (cnt + 15) >> 4;
    const int ent_incl = waveInclusiveScan(cnt);
    const int blk_incl = waveInclusiveScan(nb_mine);
    const int total = __builtin_amdgcn_readlane(ent_incl, 63);
    const int nblk = __builtin_amdgcn_readlane(blk_incl, 63);
    slots += total;
    const int nbatch = (nblk + G - 1) / G;
    const int ent_first = ent_incl - cnt;
#pragma unroll
    for (int j = 0; j < KPW; ++j) {
      const int kk = wave + j * ALLW;
      int base = __shfl(ent_first, kk & 63, kWave);
#pragma unroll
      for (int seg = 0; seg < NSEG; ++seg) {
        const unsigned long long b = __ballot(idx[j][seg] >= 0);
        if (idx[j][seg] >= 0)
          s_ent[base + __popcll(b & lt_mask)] = ((uint32_t)idx[j][seg] << 8) | (uint32_t)own[j][seg];
        base += __popcll(b);
      }
    }
    // lane kk of the wave that scanned offset kk cuts its list into blocks
    if (lane < KC && (lane % ALLW) == wave) {
      const int first_blk = blk_incl - nb_mine;
      for (int b = 0; b < nb_mine; ++b) {
        const int left = cnt - 16 * b;
        s_blk[first_blk + b] = ((uint32_t)lane << 24) | ((uint32_t)(ent_first + 16 * b) << 8) |
                               (uint32_t)(left < 16 ? left : 16);
      }
    }
    if (wave == WAVES && nblk > 0) {
      // empty blocks that fill the last batch: offset and position of the last entry
      const int last_k = 63 - __builtin_clzll(__ballot(cnt > 0));
      if (lane < nbatch * G - nblk)
        s_blk[nblk + lane] = ((uint32_t)last_k << 24) | ((uint32_t)(total - 1) << 8);
    }
    __syncthreads();

    // B: the round a batch belongs to follows from the first entry of its first block
    const int last_round =
        nblk > 0 ? (int)((s_blk[(nbatch - 1) * G] >> 8) & 0xffffu) / STEP : 0;
    if (fetcher) {
      if (nblk > 0) {
        for (int round = 0; round <= last_round; ++round) {
          u32x4 piece[PT];
#pragma unroll
          for (int i = 0; i < PT; ++i) {
            const int p = ftid + i * 64 * FW;
            int ci = round * STEP + p / PPR;
            ci = ci < total ? ci : total - 1;
            const uint32_t src = s_ent[ci] >> 8;
            const int at = (p % PPR) * 16;
            piece[i] = *reinterpret_cast<const u32x4 *>(
                at < rows.row_bytes ? a_bytes + (size_t)src * rows.row_bytes + at
                                    : reinterpret_cast<const char *>(kZeroRow));
          }
          if (round > 0) __syncthreads();  // the multiplying waves have left the stage
#pragma unroll
          for (int i = 0; i < PT; ++i) {
            const int p = ftid + i * 64 * FW;
            *reinterpret_cast<u32x4 *>(&s_stage[(p / PPR) * STAGE_STRIDE + (p % PPR) * 16]) = piece[i];
          }
          __syncthreads();
        }
      }
    } else if (nblk > 0) {
      vec8 wnext[G][KB][NB];
      uint32_t dnext[G];
      int k_held[G];  // offset whose fragments slot g holds: a dense offset fills several
                      // batches in a row and its fragments are fetched once
#pragma unroll
      for (int g = 0; g < G; ++g) k_held[g] = -1;
      auto fetch_batch = [&](int b0) {
        const uint32_t dv = s_blk[b0 + (lane & (G - 1))];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          dnext[g] = (uint32_t)__builtin_amdgcn_readlane((int)dv, g);
          const int kk = (int)(dnext[g] >> 24);
          // (single-block batches only: with several slots the branch costs the other
          // instances more than the saved loads)
          if (G > 1 || kk != k_held[g]) {
            k_held[g] = kk;
            const char *bk = b_base + (size_t)(kc + kk) * kBytesPerOffset;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
              for (int nb = 0; nb < NB; ++nb)
                wnext[g][kb][nb] = *reinterpret_cast<const vec8 *>(bk + (nb * KB + kb) * 1024);
          }
        }
      };
      fetch_batch(0);
      __syncthreads();  // round 0 is staged
      int round = 0;
      for (int bt = 0; bt < nbatch; ++bt) {
        vec8 wcur[G][KB][NB];
        uint32_t dcur[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          dcur[g] = dnext[g];
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) wcur[g][kb][nb] = wnext[g][kb][nb];
        }
        if (bt + 1 < nbatch) fetch_batch((bt + 1) * G);
        // the stage moves on when the batch starts past the current round
        while ((int)((dcur[0] >> 8) & 0xffffu) >= (round + 1) * STEP) {
          __syncthreads();
          __syncthreads();
          ++round;
        }
        const int stage_first = round * STEP;
        vec8 afr[G][KB];
        int acc_row[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int first = (int)((dcur[g] >> 8) & 0xffffu);
          const int n = (int)(dcur[g] & 0xffu);
          const int e = first + (pair < n ? pair : 0);
          const uint32_t ent = s_ent[e];
          acc_row[g] = pair < n ? (int)(ent & 0xffu) : TR;
          const char *arow = stage_lane + (e - stage_first) * STAGE_STRIDE;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
            afr[g][kb] = *reinterpret_cast<const vec8 *>(arow + kb * 64);
          if constexpr (kPartialFragment) {
            // the row ends after Q channels: the lanes of the upper quads would read the next
            // staged row; they multiply zero filter fragments, and zero keeps a NaN there out
            if (quad * E::kVec >= Q) afr[g][0] = vec8{};
          }
        }
        float4v prod[G][NB];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            prod[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
              prod[g][nb] = E::mfma(wcur[g][kb][nb], afr[g][kb], prod[g][nb]);
          }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          char *dst = acc_lane + acc_row[g] * (ACC_STRIDE * 4);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            // lane holds result columns 16*nb + 4*quad + (0..3) of its pair
            float4v old = *reinterpret_cast<float4v *>(dst + nb * 64);
            old += prod[g][nb];
            *reinterpret_cast<float4v *>(dst + nb * 64) = old;
          }
        }
      }
      // rounds the fetching wave staged beyond the last batch cannot exist:
      // last_round is the round of the last batch
    }
    __syncthreads();
  }
  constexpr int VALS = 16 / (int)sizeof(S);  // result values per 16-byte store
  for (int i = tid; i < TR * C / VALS; i += NT) {
    const int rr = i / (C / VALS);
    const int c0 = (i % (C / VALS)) * VALS;
    if (r0 + rr >= R) break;
    S tmp[VALS];
#pragma unroll
    for (int e = 0; e < VALS; ++e) E::store(&tmp[e], activated(s_acc[rr * ACC_STRIDE + c0 + e], rows.relu));
    storeColumns<E>(result + (size_t)(r0 + rr) * rows.c, col_group * C + c0, rows.c, tmp);
  }
  if constexpr (!SRC::kSegments) {
    if (tid == 0 && blockIdx.y == 0) source.filled[blockIdx.x] = slots;
  }
}

constexpr uint32_t kNoRow = 0x80000000u;  // byte offset of a partner that is not there

// The gathered tensor as a buffer of `bytes` (below 2^31) for loads that answer zero behind it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rowsBuffer(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// ---- MFMA gather convolution, tall tiles -------------------------------------------------
//
// What a thinly filled offset costs a tile is its filter: every (tile, offset) piece that holds a pair
// loads W[k] from L2 (16 KB for 64 columns of 128 channels of a 2-byte type, 12.8 GB in all at
// 5x5x5, 400 000 rows, 128 -> 128, where the kernel above takes 715 us) for as many pairs as the tile's
// rows have there.  Here a tile has 256 result rows by 64 columns, two workgroups a CU, which is what
// LDS holds fp32 sums for when nothing else of the tile lies there whole: the entries of up to
// max_blocks blocks of 16 pairs and two rounds of gathered rows.  The rest travels in registers:
//   fetching waves     request the rows of round r + ahead and write those of round r to LDS, their
//                      pieces of 16 bytes permuted by row, so that the 16 rows of a block meet all banks;
//   multiplying waves  own 16 result columns each: per block the operand fragments from the staged
//                      rows, W[k] from registers (requested `ahead` rounds before), and a 16-byte
//                      read-modify-write of every pair's sums.  The sums of a round are updated while
//                      the next round's rows are read: both are chains of LDS round trips.
// One barrier a round.  The arithmetic and its order are those of gatherConvMfma, bit for bit.
// 715 -> 460 us at the shape above; 120 000 rows, 3x3x3, 64 -> 64: 35 -> 30.  What bounds it there: a tile's first
// rows arrive 4.7 us after its start (cuts, pairs and rows are three dependent loads), a round of two
// blocks takes about 0.4 us, and the launch lasts as long as its heaviest tile (28 us, mean 16).
// Rounds are padded to whole trips of the loops, which have one way out each: with a second one the
// compiler waits for all loads in flight at the loop's head.
//
// Tiles of 512 rows of a 2-byte type (tallTileRows) halve the filters a row costs and fill their blocks better (0.69 of
// the pairs of a block instead of 0.48 at the 5x5x5 shape).  They leave a CU one workgroup, and a round is a chain of LDS
// round trips: so eight waves multiply, as two teams that take the rounds in turn.  A team reads its round's
// rows and adds its last products while the other multiplies, and the other way round: two barriers a round of a team,
// one a round of the tile, and sums still change in the order of the blocks.
// 449 -> 360 us at the 5x5x5 shape; 409 without the teams.  Of the 360 some 60 are tiles' beginnings and ends; without
// the requests of filters and rows 317 are left, so the rest is the rounds' chains.  (Twice as many rounds under way, sums
// by LDS additions without return (2680 us), or entries of one word: none faster.)  At 256 rows teams gave 2 %.
struct TallPlan {
  int per_cu;      // workgroups a CU
  int blocks;      // blocks of 16 pairs a round
  int ahead;       // rounds whose rows and filters travel in registers
  int max_blocks;  // blocks whose entries are in LDS at once
  bool teams;      // the multiplying waves are two teams
  int multipliers; // multiplying waves
};
constexpr int kTallCols = 64;
constexpr int kTallFetchers = 4;  // fetching waves
// Two workgroups of 256 rows share a CU, but for rows of 512 bytes, of which the second would leave
// no room for a round.  (Few rows run in half of the 256, many offsets in twice as many: tallTileRows.)
constexpr int tallRows(int row_bytes) { return row_bytes >= 512 ? 512 : 256; }
// (Tiles of 128 rows take the plan of 256.)
constexpr TallPlan tallPlan(int elem_bytes, int row_bytes, int tile_rows) {
  const int rows = tile_rows == 512 ? 512 : 256;
  TallPlan p = {rows == 256 ? 2 : 1, 1, 4, 0, elem_bytes == 2 && rows == 512, 4};
  if (p.teams) p.multipliers = 8;
  p.blocks = (rows == 256 ? 4096 : 8192) / (16 * row_bytes);
  const int left = 160 * 1024 / p.per_cu - (rows + 1) * kTallCols * 4 - 2 * p.blocks * 16 * row_bytes - 256;
  p.max_blocks = left / 98 / (p.ahead * p.blocks) * (p.ahead * p.blocks);
  return p;
}
constexpr int tallThreads(int elem_bytes, int row_bytes, int tile_rows) {
  return (tallPlan(elem_bytes, row_bytes, tile_rows).multipliers + kTallFetchers) * 64;
}
constexpr int tallWavesPerSimd(int elem_bytes, int row_bytes, int tile_rows) {
  return tallPlan(elem_bytes, row_bytes, tile_rows).per_cu * tallThreads(elem_bytes, row_bytes, tile_rows) / 256;
}
// Where 16-byte piece `piece` of staged row `row` lies: piece ^ this.
constexpr int tallRowSwizzle(int row_bytes, int row) {
  return row_bytes >= 256 ? (row & 15) : (row_bytes >= 128 ? ((row >> 1) & 7) : ((row >> 2) & 3));
}

template <typename E, int Q, int C, int TR, typename SRC>
__global__ __launch_bounds__(tallThreads((int)sizeof(typename E::storage), Q * (int)sizeof(typename E::storage), TR))
    __attribute__((amdgpu_waves_per_eu(
        tallWavesPerSimd((int)sizeof(typename E::storage), Q * (int)sizeof(typename E::storage), TR),
        tallWavesPerSimd((int)sizeof(typename E::storage), Q * (int)sizeof(typename E::storage), TR))))
void gatherConvTall(const typename E::storage *A, uint32_t a_size, ConvRows rows, const typename E::storage *packedW,
                    SRC source, int R, int K, typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int ROW_BYTES = Q * (int)sizeof(S);
  constexpr TallPlan PLAN = tallPlan((int)sizeof(S), ROW_BYTES, TR);
  constexpr int MW = PLAN.multipliers;
  constexpr int FW = kTallFetchers;
  constexpr int NT = (MW + FW) * 64;
  constexpr bool kTeams = PLAN.teams;
  constexpr int TW = kTeams ? MW / 2 : MW;   // waves of a team
  constexpr int NB = C / 16 / TW;            // column blocks of a multiplying wave
  constexpr int KB = ROW_BYTES / 64;         // operand fragments per row
  constexpr int G = PLAN.blocks;
  constexpr int U = PLAN.ahead;
  constexpr int MAXB = PLAN.max_blocks;
  constexpr int ROUND = G * 16 * ROW_BYTES;
  constexpr int NI = ROUND / 1024 / FW;      // loads of a fetching wave per round
  constexpr int PPR = ROW_BYTES / 16;
  constexpr int GROUPS = C / 16;
  constexpr int ALLW = NT / 64;
  constexpr int NSEG = TR / 64;
  constexpr int KPW = 32 / ALLW;             // offsets of a row map a wave reads at once
  static_assert(ROUND % (1024 * FW) == 0 && NI >= 1, "a round splits evenly over the fetching waves");
  static_assert(MAXB >= TR / 16, "an offset's pairs fit");

  __shared__ __attribute__((aligned(1024))) char s_stage[2 * ROUND];
  __shared__ __attribute__((aligned(256))) float s_acc[(TR + 1) * C];
  __shared__ uint32_t s_src[MAXB * 16];  // where the gathered row begins; kNoRow: no pair
  __shared__ u16 s_row[MAXB * 16];       // result row in the tile; TR: no pair
  __shared__ u16 s_k[MAXB];              // offset of a block
  __shared__ int s_count[SRC::kSegments ? 1 : KPW * ALLW];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool fetcher = wave >= MW;
  const int tiles_per_xcd = gridDim.x >> 3;  // neighbouring tiles on one XCD, as above
  const int tile = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  const int r0 = tile * TR;
  if constexpr (!SRC::kSegments) {
    if (notWanted(source.run_if)) return;
  }
  if (r0 >= R) {
    if constexpr (!SRC::kSegments) {
      if (tid == 0 && blockIdx.y == 0) source.filled[blockIdx.x] = 0;
    }
    return;
  }
  int slots = 0;  // filled map slots of this tile
  // lane l: the piece of offset kc + l
  int first = 0, count = 0;
  auto look_up = [&](int kc) {
    if constexpr (SRC::kSegments) {
      const int k_mine = kc + lane < K ? kc + lane : K - 1;
      const int32_t *const cut = source.cuts + (size_t)k_mine * source.cut_stride + tile;
      first = cut[0];
      count = cut[1] - first;
      count = count < 0 ? 0 : (count > TR ? TR : count);
      if (kc + lane >= K || source.counts.n[k_mine] <= 0) count = 0;
    }
  };
  // (requested ahead of the clearing, which takes as long)
  bool in_order = true;
  unsigned long long verdict = 0;
  if constexpr (SRC::kSegments) verdict = *source.verdict;
  look_up(0);
  for (int i = tid; i < (TR + 1) * C / 4; i += NT) reinterpret_cast<float4v *>(s_acc)[i] = float4v{0.f, 0.f, 0.f, 0.f};
  const int col_group = blockIdx.y;
  if constexpr (SRC::kSegments) {
    in_order = verdict != source.ticket;
    if (!in_order && source.leave_if_unordered) return;
    if (!in_order) {
      __syncthreads();
      const int columns = rows.c - col_group * C;
      scanAllPairsForTile<E, NT>(A, rows.q, rows.row_bytes, source, K, r0, r0 + TR < R ? r0 + TR : R,
                                 columns < C ? columns : C, col_group * C, s_acc, C);
    }
  }

  const int pair = lane & 15;
  const int quad = lane >> 4;
  const __amdgpu_buffer_rsrc_t a_rows = rowsBuffer(A, a_size);
  const char *const b_base = reinterpret_cast<const char *>(packedW) +
                             ((size_t)(col_group * GROUPS + wave % TW * NB) * KB * 64 + lane) * 16;
  const uint32_t bytes_per_offset = (uint32_t)(rows.c_padded / 16) * KB * 1024;  // packed W[k]

  for (int kc = 0; kc < (in_order ? K : 0);) {
    // A: the entries of as many offsets as the lists have room for
    if (kc > 0) look_up(kc);
    // (row map: its slots of kMapOffsets offsets, wave w those of the offsets w, w + ALLW, ...)
    int partners[KPW][NSEG];
    if constexpr (!SRC::kSegments) {
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int k = kc + wave + j * ALLW < K ? kc + wave + j * ALLW : K - 1;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          const int r = r0 + seg * 64 + lane;
          partners[j][seg] = source.map[(size_t)k * R + (r < R ? r : R - 1)];
        }
      }
#pragma unroll
      for (int j = 0; j < KPW; ++j)
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) asm volatile("" : "+v"(partners[j][seg]));
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        int c = 0;
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          if (kc + wave + j * ALLW >= K || r0 + seg * 64 + lane >= R) partners[j][seg] = -1;
          c += __popcll(__ballot(partners[j][seg] >= 0));
        }
        if (lane == 0) s_count[wave + j * ALLW] = c;
      }
      __syncthreads();
      count = lane < KPW * ALLW ? s_count[lane < KPW * ALLW ? lane : 0] : 0;
    }
    constexpr int kAtOnce = SRC::kSegments ? 64 : KPW * ALLW;  // offsets looked up
    const int blk_end = waveInclusiveScan((count + 15) >> 4);
    const int taken = __popcll(__ballot(blk_end <= MAXB && lane < kAtOnce && kc + lane < K));
    const int n_blocks = __builtin_amdgcn_readlane(blk_end, taken - 1);
    const int n_rounds = ((n_blocks + G - 1) / G + U - 1) / U * U;
    const int blk_first = blk_end - ((count + 15) >> 4);
    if constexpr (!SRC::kSegments) {
      slots += __builtin_amdgcn_readlane(waveInclusiveScan(count), taken - 1);
      // no pair, where none is written behind the next barrier
      for (int e = tid; e < n_rounds * G * 16; e += NT) {
        s_src[e] = kNoRow;
        s_row[e] = (u16)TR;
        if ((e & 15) == 0) s_k[e >> 4] = (u16)(kc + taken - 1);
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        const int kk = wave + j * ALLW;
        int at = __shfl(blk_first, kk, kWave) * 16;
        const int last = __shfl(blk_end, kk, kWave);
        if (kk >= taken) continue;
        for (int b = at / 16 + lane; b < last; b += kWave) s_k[b] = (u16)(kc + kk);
#pragma unroll
        for (int seg = 0; seg < NSEG; ++seg) {
          const unsigned long long m = __ballot(partners[j][seg] >= 0);
          if (partners[j][seg] >= 0) {
            const int e = at + __popcll(m & ((1ull << lane) - 1ull));
            s_src[e] = (uint32_t)partners[j][seg] * (uint32_t)rows.row_bytes;
            s_row[e] = (u16)(seg * 64 + lane);
          }
          at += __popcll(m);
        }
      }
    } else {
    // block b belongs to the first lane whose blocks end behind it
    constexpr int PER = (MAXB * 16 + NT - 1) / NT;  // entries a thread
    int own_row[PER], partner[PER], k_of[PER];
    bool there[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int b = (tid + u * NT) >> 4;
      int at = 0;
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        if (__shfl(blk_end, at + step - 1, kWave) <= b) at += step;
      at = at < taken ? at : taken - 1;
      const int i = (b - __shfl(blk_first, at, kWave)) * 16 + (lane & 15);
      const int pairs_there = __shfl(count, at, kWave);  // (outside the condition: all lanes take part)
      const bool live = b < n_blocks && i < pairs_there;
      int p = __shfl(first, at, kWave) + (live ? i : 0);
      p = p < 0 ? 0 : (p < source.L ? p : source.L - 1);
      const int32_t *const list = source.pairs + (size_t)(kc + at) * 2 * source.L;
      own_row[u] = list[(size_t)source.row_col * source.L + p];
      partner[u] = list[(size_t)source.src_col * source.L + p];
      there[u] = live;
      k_of[u] = kc + at;
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) asm volatile("" : "+v"(own_row[u]), "+v"(partner[u]));
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + u * NT;
      if (e < MAXB * 16) {
        s_src[e] = there[u] ? (uint32_t)partner[u] * (uint32_t)rows.row_bytes : kNoRow;
        s_row[e] = there[u] ? (u16)((own_row[u] - r0) & (TR - 1)) : (u16)TR;
        if ((lane & 15) == 0) s_k[e >> 4] = (u16)k_of[u];
      }
    }
    }
    kc += taken;
    __syncthreads();
    if (n_blocks == 0) continue;
    // B
    if (fetcher) {
      const int ftid = tid - MW * 64;
      u32x4 piece[U][NI];
      auto request_round = [&](int round, u32x4 (&to)[NI]) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int slot = ftid + j * 64 * FW;
          const uint32_t from = s_src[round * G * 16 + slot / PPR];
          const uint32_t at = slot % PPR * 16 < rows.row_bytes ? (uint32_t)(slot % PPR * 16) : kNoRow;
          to[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                a_rows, __builtin_elementwise_add_sat(from, at), 0, 0));
        }
      };
#pragma unroll
      for (int j = 0; j < U; ++j) {
        request_round(j, piece[j]);
        asm volatile("" ::: "memory");  // (in this order: the loop below waits for the oldest)
      }
      for (int r = 0; r < n_rounds; r += U) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
          char *const stage = s_stage + ((r + j) & 1) * ROUND;
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const int slot = ftid + i * 64 * FW;
            const int row = slot / PPR;
            *reinterpret_cast<u32x4 *>(stage + row * ROW_BYTES +
                                       ((slot % PPR) ^ tallRowSwizzle(ROW_BYTES, row & 15)) * 16) = piece[j][i];
          }
          request_round(r + j + U < n_rounds ? r + j + U : n_rounds - 1, piece[j]);
          ldsBarrier();  // round r + j is there, and nobody reads the round before any more
        }
      }
      if constexpr (kTeams) {  // (the phases behind the last round's first)
        ldsBarrier();
        ldsBarrier();
      }
    } else if (col_group * C + wave % TW * NB * 16 >= rows.c) {
      // no result column of this wave's: its part of the barriers (the other workgroup gets its CU's pipes: fp32
      // 64 -> 96, 2x2x2 stride 2 of 200 000 rows, 74 -> 70 us)
      for (int r = 0; r < n_rounds; r += U) {
#pragma unroll
        for (int j = 0; j < U; ++j) ldsBarrier();
      }
      if constexpr (kTeams) {
        ldsBarrier();
        ldsBarrier();
      }
    } else if constexpr (kTeams) {
      constexpr int UT = U / 2;  // of a team's rounds, whose filters travel in registers
      const int team = wave / TW, part = wave % TW;
      vec8 w[UT][G][KB][NB];
      auto request_filters = [&](const int (&ks)[G], vec8 (&to)[G][KB][NB]) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const char *const bk = b_base + (size_t)__builtin_amdgcn_readfirstlane(ks[g]) * bytes_per_offset;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) to[g][kb][nb] = *reinterpret_cast<const vec8 *>(bk + (nb * KB + kb) * 1024);
        }
      };
      // (round t of the team)
      auto offsets_of = [&](int t, int (&ks)[G]) {
        const int r = t * 2 + team < n_rounds ? t * 2 + team : n_rounds - 1;
#pragma unroll
        for (int g = 0; g < G; ++g) ks[g] = s_k[r * G + g];
      };
      int ks[G], own[G];
#pragma unroll
      for (int j = 0; j < UT; ++j) {
        offsets_of(j, ks);
        request_filters(ks, w[j]);
        asm volatile("" ::: "memory");
      }
      offsets_of(UT, ks);
      float4v prod[G][NB];
      // one block after the other, since blocks of different offsets may meet in a row
      auto add_block = [&](int g) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          // lane holds result columns 4 * piece + (0..3) of its pair
          const int piece = (part * NB + nb) * 4 + quad;
          float4v *const sum = reinterpret_cast<float4v *>(s_acc) + own[g] * (C / 4) + (piece ^ (own[g] & 15));
          float4v old = *sum;
          old += prod[g][nb];
          *sum = old;
        }
      };
#pragma unroll
      for (int g = 0; g < G; ++g) own[g] = TR;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) prod[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
      if (team == 1) ldsBarrier();
      const char *const stage = s_stage + team * ROUND;
      for (int t = 0; t < n_rounds / 2; t += UT) {
#pragma unroll
        for (int j = 0; j < UT; ++j) {
          ldsBarrier();  // the round is there, and the other team has added the round between
          vec8 a[G][KB];
#pragma unroll
          for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
              a[g][kb] = *reinterpret_cast<const vec8 *>(stage + (g * 16 + pair) * ROW_BYTES +
                                                         (((kb * 4 + quad) ^ tallRowSwizzle(ROW_BYTES, pair)) * 16));
            add_block(g);
          }
#pragma unroll
          for (int g = 0; g < G; ++g) own[g] = s_row[(((t + j) * 2 + team) * G + g) * 16 + pair];
          ldsBarrier();
#pragma unroll
          for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) prod[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
              for (int nb = 0; nb < NB; ++nb) prod[g][nb] = E::mfma(w[j][g][kb][nb], a[g][kb], prod[g][nb]);
          }
          request_filters(ks, w[j]);
          offsets_of(t + j + UT + 1, ks);
        }
      }
      ldsBarrier();
#pragma unroll
      for (int g = 0; g < G; ++g) add_block(g);
      if (team == 0) ldsBarrier();
    } else {
      vec8 w[U][G][KB][NB];
      // filters of a round whose blocks have the offsets ks
      auto request_filters = [&](const int (&ks)[G], vec8 (&to)[G][KB][NB]) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const char *const bk = b_base + (size_t)__builtin_amdgcn_readfirstlane(ks[g]) * bytes_per_offset;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) to[g][kb][nb] = *reinterpret_cast<const vec8 *>(bk + (nb * KB + kb) * 1024);
        }
      };
      auto offsets_of = [&](int round, int (&ks)[G]) {
        const int r = round < n_rounds ? round : n_rounds - 1;
#pragma unroll
        for (int g = 0; g < G; ++g) ks[g] = s_k[r * G + g];
      };
      auto rows_of = [&](int round, int (&own)[G]) {
        const int r = round < n_rounds ? round : n_rounds - 1;
#pragma unroll
        for (int g = 0; g < G; ++g) own[g] = s_row[(r * G + g) * 16 + pair];
      };
      int ks[G], own[G], own_next[G];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        offsets_of(j, ks);
        request_filters(ks, w[j]);
        asm volatile("" ::: "memory");
      }
      offsets_of(U, ks);
      float4v prod[G][NB];
      // the products of the round before go to their sums while this round's rows are read from LDS:
      // one block after the other, since blocks of different offsets may meet in a row
      auto add_block = [&](int g) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          // lane holds result columns 4 * piece + (0..3) of its pair
          const int piece = (wave * NB + nb) * 4 + quad;
          float4v *const sum = reinterpret_cast<float4v *>(s_acc) + own[g] * (C / 4) + (piece ^ (own[g] & 15));
          float4v old = *sum;
          old += prod[g][nb];
          *sum = old;
        }
      };
#pragma unroll
      for (int g = 0; g < G; ++g) own[g] = TR;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) prod[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
      rows_of(0, own_next);
      for (int r = 0; r < n_rounds; r += U) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
          ldsBarrier();
          const char *const stage = s_stage + ((r + j) & 1) * ROUND;
          vec8 a[G][KB];
#pragma unroll
          for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
              a[g][kb] = *reinterpret_cast<const vec8 *>(stage + (g * 16 + pair) * ROW_BYTES +
                                                         (((kb * 4 + quad) ^ tallRowSwizzle(ROW_BYTES, pair)) * 16));
            add_block(g);
          }
#pragma unroll
          for (int g = 0; g < G; ++g) own[g] = own_next[g];
          rows_of(r + j + 1, own_next);
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
              prod[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int kb = 0; kb < KB; ++kb) prod[g][nb] = E::mfma(w[j][g][kb][nb], a[g][kb], prod[g][nb]);
            }
          request_filters(ks, w[j]);
          offsets_of(r + j + U + 1, ks);
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) add_block(g);
    }
    __syncthreads();
  }
  __syncthreads();
  constexpr int VALS = 16 / (int)sizeof(S);
  for (int i = tid; i < TR * C / VALS; i += NT) {
    const int rr = i / (C / VALS);
    const int c0 = (i % (C / VALS)) * VALS;
    if (r0 + rr >= R) break;
    S tmp[VALS];
#pragma unroll
    for (int q = 0; q < VALS / 4; ++q) {
      const int piece = c0 / 4 + q;
      const float4v v = reinterpret_cast<const float4v *>(s_acc)[rr * (C / 4) + (in_order ? piece ^ (rr & 15) : piece)];
#pragma unroll
      for (int e = 0; e < 4; ++e) E::store(&tmp[q * 4 + e], activated(v[e], rows.relu));
    }
    storeColumns<E>(result + (size_t)(r0 + rr) * rows.c, col_group * C + c0, rows.c, tmp);
  }
  if constexpr (!SRC::kSegments) {
    if (tid == 0 && blockIdx.y == 0) source.filled[blockIdx.x] = slots;
  }
}

// ---- MFMA gather convolution, one free-running wavefront per tile ---------------------
//
// The kernel above spends a tile's life waiting: cut positions, then pairs, then
// gathered rows round by round behind barriers, then a filter slice from L2 for every
// thinly filled offset, with two tiles a CU to overlap it all.  For results of up to 32
// columns a tile of 128 result rows fits a single wavefront that never meets a barrier:
// its fp32 accumulator tile and one 16-row stage slot are all the LDS it needs, so
// seven tiles share a CU, a layer of a few hundred thousand rows is resident at once,
// and what the wave waits for is hidden by its own requests running ahead in register
// rings:
//   unit      = up to 16 pairs of one offset, walked in offset order;
//   t + 10    the unit's pairs are requested (lane l: pair l % 16);
//   t + 5     its gathered rows (row-contiguous 16-byte pieces) and the offset's filter
//             fragments are requested;
//   t         rows go through the LDS slot (written row-major, read as MFMA operand
//             fragments), all column blocks are multiplied and the products added to the
//             pairs' fp32 rows, read from and written back to LDS 16 bytes a lane.
// Requests are unconditional (clamped addresses) so that the number of loads in flight
// at every point of the loop is fixed.  It reads pair lists only (SegmentSource).
// Measured against the kernel above on 120 000 rows with 2.2 pairs a row: 32 -> 32
// channels 26 us against 32 us; at 64 result columns (two waves a tile, 32 columns
// each) it loses, 43 us against 41 us, and is not used.
// WHOLE: rows and results of exactly Q and C channels, with their lengths as constants (the same
// layers with lengths from the arguments: 16 -> 16 channels 30.8 against 28.6 us, 32 -> 32 35 against 32).
constexpr int kWaveTileRows = 128;
constexpr bool waveKernelShape(int elem_bytes, int Q, int C) {
  const int chunk = elem_bytes == 4 ? 16 : 32;
  return C <= 32 && Q * elem_bytes <= 256 && ((Q + chunk - 1) / chunk) * (C / 16) <= 8;
}
template <typename E, int Q, int C, bool WHOLE>
__global__ __launch_bounds__(64) void gatherConvWave(
    const typename E::storage *A, ConvRows lengths, const typename E::storage *packedW, SegmentSource source,
    int R, int K, typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int NB = C / 16;                            // column blocks
  constexpr int KB = (Q + E::kChunk - 1) / E::kChunk;
  constexpr bool kPartialFragment = Q < E::kChunk;
  constexpr int TR = kWaveTileRows;
  constexpr int ACC_STRIDE = C + 4;
  constexpr int ROW_BYTES = Q * (int)sizeof(S);
  const ConvRows conv = WHOLE ? ConvRows{Q, ROW_BYTES, C, C, lengths.relu} : lengths;
  constexpr int STAGE_STRIDE = ROW_BYTES + 16;
  constexpr int PPR = ROW_BYTES / 16;                   // 16-byte pieces per row
  constexpr int RL = (16 * PPR + 63) / 64;              // wave-loads per unit of rows
  constexpr int EPL = 64 / PPR >= 16 ? 16 : 64 / PPR;   // rows per wave-load
  constexpr int NE = 12;   // pair ring (units) = units per trip of the unrolled loop
  constexpr int NR = 6;    // row and filter ring (units)
  constexpr int AHEAD_ROWS = 5;
  constexpr int AHEAD_PAIRS = 10;
  static_assert(PPR >= 2 && PPR <= 32 && AHEAD_ROWS < NR && AHEAD_PAIRS < NE && NE % NR == 0, "ring sizes");
  constexpr int ACC_QUADS = (TR + 1) * ACC_STRIDE / 4;

  __shared__ __attribute__((aligned(16))) float s_acc[(TR + 1) * ACC_STRIDE];
  __shared__ __attribute__((aligned(16))) char s_stage[16 * STAGE_STRIDE];

  const int lane = threadIdx.x;
  const int tiles_per_xcd = gridDim.x >> 3;  // neighbouring tiles on one XCD
  const int tile = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  const int r0 = tile * TR;
  if (r0 >= R) return;

  // this tile's piece of every offset's list (lane l: offsets l and l + 64)
  const unsigned long long verdict = *source.verdict;
  int piece_first[2] = {0, 0}, piece_count[2] = {0, 0};
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    const int k = lane + 64 * o;
    if (k < K) {
      const int32_t *c = source.cuts + (size_t)k * source.cut_stride + tile;
      piece_first[o] = c[0];
      piece_count[o] = c[1];
    }
  }
#pragma unroll 8
  for (int i = lane; i < ACC_QUADS; i += 64)
    reinterpret_cast<float4v *>(s_acc)[i] = float4v{0.f, 0.f, 0.f, 0.f};

  constexpr int VALS = 16 / (int)sizeof(S);
  auto write_out = [&]() {
    for (int i = lane; i < TR * C / VALS; i += 64) {
      const int rr = i / (C / VALS);
      const int c0 = (i % (C / VALS)) * VALS;
      if (r0 + rr >= R) break;
      S tmp[VALS];
#pragma unroll
      for (int e = 0; e < VALS; ++e) E::store(&tmp[e], activated(s_acc[rr * ACC_STRIDE + c0 + e], conv.relu));
      storeColumns<E>(result + (size_t)(r0 + rr) * conv.c, c0, conv.c, tmp);
    }
  };
  if (verdict == source.ticket) {
    if (source.leave_if_unordered) return;
    // lists out of order: every pair of every offset is looked at
    scanAllPairsForTile<E, 64>(A, conv.q, conv.row_bytes, source, K, r0, r0 + TR < R ? r0 + TR : R,
                               conv.c, 0, s_acc, ACC_STRIDE);
    write_out();
    return;
  }
  unsigned long long has[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    int c = piece_count[o] - piece_first[o];
    c = c < 0 ? 0 : (c > TR ? TR : c);
    if (lane + 64 * o >= K) c = 0;
    piece_count[o] = c;
    has[o] = __ballot(c > 0);
  }
  // first offset above `after` that has pairs in this tile, or 128
  auto next_offset = [&](int after) {
    const int from = after + 1;
    const unsigned long long lo = from < 64 ? (has[0] & (~0ull << from)) : 0ull;
    if (lo) return (int)__builtin_ctzll(lo);
    const unsigned long long hi = from <= 64 ? has[1] : (from < 128 ? (has[1] & (~0ull << (from - 64))) : 0ull);
    if (hi) return 64 + (int)__builtin_ctzll(hi);
    return 128;
  };
  auto of = [&](const int (&v)[2], int k) {
    const int a = __builtin_amdgcn_readlane(v[0], k & 63), b = __builtin_amdgcn_readlane(v[1], k & 63);
    return k < 64 ? a : b;
  };
  // the walk over units: offset, first pair and pair count of the unit a request is made for
  int walk_k = next_offset(-1);
  int walk_left = walk_k < 128 ? of(piece_count, walk_k) : 0;
  int walk_at = walk_k < 128 ? of(piece_first, walk_k) : 0;
  int unit_k[NE], unit_at[NE], unit_n[NE];
  auto next_unit = [&](int &k, int &at, int &n) {
    k = walk_k;
    at = walk_at;
    n = walk_left < 16 ? walk_left : 16;
    if (walk_k < 128) {
      walk_left -= n;
      walk_at += n;
      if (walk_left <= 0) {
        walk_k = next_offset(walk_k);
        walk_left = walk_k < 128 ? of(piece_count, walk_k) : 0;
        walk_at = walk_k < 128 ? of(piece_first, walk_k) : 0;
      }
    }
  };

  const char *a_bytes = reinterpret_cast<const char *>(A);
  const char *b_base = reinterpret_cast<const char *>(packedW) + (size_t)lane * 16;
  const uint32_t kBytesPerOffset = (uint32_t)(C / 16) * KB * 64 * 16;
  const int pair = lane & 15;
  const int quad = lane >> 4;
  char *acc_lane = reinterpret_cast<char *>(s_acc) + 4 * quad * 4;
  char *stage = s_stage;

  // Rows of up to 64 bytes are loaded by the lane that multiplies them, 16 bytes of its own
  // pair's row (the 16 rows of a unit are 16 cache lines either way); longer rows are
  // fetched row by row, half as many lines a load, and turned into fragments by the LDS slot.
  constexpr bool kDirectRows = ROW_BYTES <= 64;
  int pair_row[NE], pair_src[NE];
  u32x4 rows[NR][RL];
  vec8 w[NR][KB][NB];

  auto request_pairs = [&](int slot) {
    next_unit(unit_k[slot], unit_at[slot], unit_n[slot]);
    const int k = unit_k[slot] < K ? unit_k[slot] : 0;
    int p = unit_at[slot] + pair;
    p = p < 0 ? 0 : (p < source.L ? p : source.L - 1);
    const int32_t *list = source.pairs + (size_t)k * 2 * source.L;
    pair_row[slot] = list[(size_t)source.row_col * source.L + p];
    pair_src[slot] = list[(size_t)source.src_col * source.L + p];
    // The requests must stay where they are written, far ahead of their use: nothing that
    // may touch memory moves across this point, so the compiler cannot sink the loads
    // towards the instructions that consume them (and no register is named, so nothing
    // is waited for here).
    asm volatile("" ::: "memory");
  };
  auto request_rows = [&](int pslot, int rslot) {
    const int n = unit_n[pslot];
    const int k = unit_k[pslot] < K ? unit_k[pslot] : 0;
    if constexpr (kDirectRows) {
      static_assert(!kDirectRows || (RL == 1 && KB == 1), "one fragment a row");
      int g = pair_src[pslot];
      if (pair >= n || (unsigned)g >= (unsigned)source.n_src) g = 0;
      // (a lane beyond the row's channels reads the row of zeros)
      const char *from = quad * 16 < conv.row_bytes ? a_bytes + (size_t)g * conv.row_bytes + quad * 16
                                                    : reinterpret_cast<const char *>(kZeroRow);
      rows[rslot][0] = *reinterpret_cast<const u32x4 *>(from);
    } else {
#pragma unroll
      for (int h = 0; h < RL; ++h) {
        const int e = lane / PPR + EPL * h;  // which pair's row this lane fetches a piece of
        int g = __shfl(pair_src[pslot], e & 15, kWave);
        if (e >= n || (unsigned)g >= (unsigned)source.n_src) g = 0;
        const int at = (lane % PPR) * 16;
        rows[rslot][h] = *reinterpret_cast<const u32x4 *>(
            at < conv.row_bytes ? a_bytes + (size_t)g * conv.row_bytes + at
                                : reinterpret_cast<const char *>(kZeroRow));
      }
    }
    const char *bk = b_base + (size_t)k * kBytesPerOffset;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        w[rslot][kb][nb] = *reinterpret_cast<const vec8 *>(bk + (nb * KB + kb) * 1024);
    asm volatile("" ::: "memory");
  };
  auto multiply = [&](int pslot, int rslot) {
    const int n = unit_n[pslot];
    const int acc_row = pair < n ? ((pair_row[pslot] - r0) & (TR - 1)) : TR;
    char *dst = acc_lane + acc_row * (ACC_STRIDE * 4);
    // (products summed from zero, then added: the arithmetic of the kernel above, so the
    // two give the same bits)
    float4v acc[NB], prod[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      acc[nb] = *reinterpret_cast<float4v *>(dst + nb * 64);
      prod[nb] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    vec8 afr[KB];
    if constexpr (kDirectRows) {
      afr[0] = __builtin_bit_cast(vec8, rows[rslot][0]);
    } else {
#pragma unroll
      for (int h = 0; h < RL; ++h) {
        const int e = lane / PPR + EPL * h;
        if (16 * PPR >= 64 || lane < 16 * PPR)
          *reinterpret_cast<u32x4 *>(stage + e * STAGE_STRIDE + (lane % PPR) * 16) = rows[rslot][h];
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        afr[kb] = *reinterpret_cast<const vec8 *>(stage + pair * STAGE_STRIDE + kb * 64 + quad * 16);
      if constexpr (kPartialFragment) {
        if (quad * E::kVec >= Q) afr[0] = vec8{};
      }
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) prod[nb] = E::mfma(w[rslot][kb][nb], afr[kb], prod[nb]);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      acc[nb] += prod[nb];
      *reinterpret_cast<float4v *>(dst + nb * 64) = acc[nb];
    }
  };

#pragma unroll
  for (int u = 0; u < AHEAD_PAIRS; ++u) request_pairs(u);
#pragma unroll
  for (int u = 0; u < AHEAD_ROWS; ++u) request_rows(u, u);
  bool more = unit_k[0] < 128;
  while (more) {
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      // unit t = t0 + u: pair slot u, row slot u % NR
      if (more) {
        request_pairs((u + AHEAD_PAIRS) % NE);
        request_rows((u + AHEAD_ROWS) % NE, (u + AHEAD_ROWS) % NR);
        multiply(u, u % NR);
        more = unit_k[(u + 1) % NE] < 128;
      }
    }
  }
  write_out();
}

// ---- MFMA gather convolution for dense rulebooks -------------------------------
//
// When most rows of a tile have a partner at most offsets, compacting pairs buys
// little and the fp32 accumulate in LDS (a 16-byte read-modify-write per lane and
// 16 result columns, on arbitrary rows: bank conflicts) is what the kernels above
// spend their time on.  Here a wave owns groups of 16 result rows and accumulates them
// in registers over all offsets: no accumulator traffic at all.  Two kernels, by the length of a
// gathered row: gatherConvDense up to 64 bytes, gatherConvDenseStaged above.
//
// Rows are buffer loads: the row map holds byte offsets, a lane without a partner holds one
// behind the tensor's end, and the hardware answers it with zeros without going to memory.
// Both kernels multiply rows of zeros for the partners that are not there, which is nothing as long
// as the filter is finite.  An offset whose filter is not (packFilter says so) is taken out of the
// walk and multiplied by itself, its products added to the rows that have a partner there only.
constexpr int kDenseChunk = 27;      // offsets whose row-map slice is resident in LDS at once
constexpr int kDenseMapBatch = 14;   // loads in flight per thread while a tile's row map is read
constexpr int kDenseRows = 128;      // of a tile
constexpr int kDenseThreads = 256;
constexpr int kDenseGroups = kDenseRows / 16;
static_assert(kDenseChunk <= 32, "a chunk's offsets in one mask");

// A tile's slice of the row map for a chunk of offsets.
struct DenseMap {
  uint32_t at[kDenseChunk][kDenseRows];  // where the partner row of (offset in chunk, tile row) begins, or kNoRow
  int first[kDenseChunk], count[kDenseChunk];
  int finite[kDenseChunk];       // the offset's filter holds no infinity and no NaN
  uint32_t groups[kDenseChunk];  // the row groups that have a partner at the offset
};

// Fills the map for the offsets [kc, kc + kn), by the whole workgroup; ends in a barrier.  Returns the filled slots of
// a MapSource that this thread has seen.
template <typename SRC>
__device__ __forceinline__ int fillDenseMap(DenseMap &map, const SRC &source, const unsigned long long *nonfinite,
                                            int row_bytes, int tile, int r0, int R, int kc, int kn, int K) {
  constexpr int TR = kDenseRows, NT = kDenseThreads;
  const int tid = threadIdx.x, lane = tid & 63;
  int slots = 0;
  if (tid < kn) map.finite[tid] = nonfinite[kc + tid] != nonfinite[K];
  if constexpr (SRC::kSegments) {
    // The pairs of an offset that fall into this tile are one piece of its list, between
    // two neighbouring entries of the cut table.
    if (tid < kn) {
      const int32_t *cut = source.cuts + (size_t)(kc + tid) * source.cut_stride + tile;
      const int first = cut[0];
      const int count = cut[1] - first;
      map.first[tid] = first;
      map.count[tid] = count < 0 ? 0 : (count > TR ? TR : count);
    }
    for (int i = tid; i < kn * TR; i += NT) (&map.at[0][0])[i] = kNoRow;
    __syncthreads();
    // a thread per (offset, pair of the piece): the partner goes to the result row's
    // position.  A thread's loads of one batch are all requested before the first is
    // used (a slot without a pair reads pair 0 of its offset and drops it).
    if (source.L > 0) {
      for (int base = tid; base < kn * TR; base += NT * kDenseMapBatch) {
        int own[kDenseMapBatch], partner[kDenseMapBatch], at[kDenseMapBatch];
#pragma unroll
        for (int u = 0; u < kDenseMapBatch; ++u) {
          const int slot = base + u * NT;
          int kk = slot / TR;
          const int q = slot % TR;
          kk = kk < kn ? kk : kn - 1;
          const bool live = slot < kn * TR && q < map.count[kk];
          int p = live ? map.first[kk] + q : 0;
          p = p < 0 ? 0 : (p < source.L ? p : source.L - 1);
          const int32_t *list = source.pairs + (size_t)(kc + kk) * 2 * source.L;
          own[u] = list[(size_t)source.row_col * source.L + p];
          partner[u] = list[(size_t)source.src_col * source.L + p];
          at[u] = live ? kk : -1;
        }
#pragma unroll
        for (int u = 0; u < kDenseMapBatch; ++u)
          if (at[u] >= 0) map.at[at[u]][(own[u] - r0) & (TR - 1)] = (uint32_t)partner[u] * (uint32_t)row_bytes;
      }
    }
  } else {
    for (int base = tid; base < kn * TR; base += NT * kDenseMapBatch) {
      int v[kDenseMapBatch];
#pragma unroll
      for (int u = 0; u < kDenseMapBatch; ++u) {
        const int slot = base + u * NT;
        int kk = slot / TR;
        kk = kk < kn ? kk : kn - 1;
        const int r = r0 + slot % TR;
        v[u] = source.map[(size_t)(kc + kk) * R + (r < R ? r : R - 1)];
        if (slot >= kn * TR || r >= R) v[u] = -1;
      }
#pragma unroll
      for (int u = 0; u < kDenseMapBatch; ++u) {
        const int slot = base + u * NT;
        if (slot < kn * TR) map.at[slot / TR][slot % TR] = v[u] >= 0 ? (uint32_t)v[u] * (uint32_t)row_bytes : kNoRow;
        slots += v[u] >= 0;
      }
    }
  }
  __syncthreads();
  // which row groups have a partner at which offsets: a thread an (offset, group)
  for (int base = 0; base < kn * kDenseGroups; base += NT) {
    const int kk = (base + tid) / kDenseGroups, group = tid % kDenseGroups;
    bool any = false;
    if (kk < kn) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 at = *reinterpret_cast<const u32x4 *>(&map.at[kk][group * 16 + q * 4]);
        any = any | (at[0] != kNoRow) | (at[1] != kNoRow) | (at[2] != kNoRow) | (at[3] != kNoRow);
      }
    }
    const unsigned long long m = __ballot(any);
    if (kk < kn && group == 0) map.groups[kk] = (uint32_t)(m >> (lane & ~(kDenseGroups - 1))) & ((1u << kDenseGroups) - 1u);
  }
  __syncthreads();
  return slots;
}

// A tile whose pair lists turned out to be out of order: fp32 rows where the row map would be, 16 columns at a time,
// every pair looked at by every workgroup.
template <typename E>
__device__ __forceinline__ void denseTileOutOfOrder(DenseMap &map, const typename E::storage *A, const ConvRows &conv,
                                                    const SegmentSource &source, int r0, int R, int K,
                                                    typename E::storage *result) {
  constexpr int TR = kDenseRows, NT = kDenseThreads, CP = 16;  // columns per pass
  static_assert(CP <= kDenseChunk, "a pass of columns fits the row map");
  float *acc = reinterpret_cast<float *>(&map.at[0][0]);
  const int r_end = r0 + TR < R ? r0 + TR : R;
  for (int c0 = 0; c0 < conv.c; c0 += CP) {
    for (int i = threadIdx.x; i < TR * CP; i += NT) acc[i] = 0.f;
    __syncthreads();
    const int columns = conv.c - c0 < CP ? conv.c - c0 : CP;
    scanAllPairsForTile<E, NT>(A, conv.q, conv.row_bytes, source, K, r0, r_end, columns, c0, acc, CP);
    for (int i = threadIdx.x; i < TR * CP; i += NT) {
      const int rr = i / CP, c = i % CP;
      if (r0 + rr < R && c < columns)
        E::store(result + (size_t)(r0 + rr) * conv.c + c0 + c, activated(acc[i], conv.relu));
    }
    __syncthreads();
  }
}

// An offset whose filter is not finite: its products, added to the rows that have a partner there only.  `at`: the
// map's entries of the wave's rows, `filter`: its first column block's fragments for lane 0.
template <typename E, int G, int NB, int KB>
__device__ __forceinline__ void addOffsetApart(float4v (&acc)[G][NB], __amdgpu_buffer_rsrc_t a_rows, const uint32_t *at_rows,
                                               const char *filter, int row_bytes) {
  typedef typename E::vec8 vec8;
  int own = threadIdx.x & 63;  // (nothing of this rare loop is worked out ahead of it and held in registers)
  asm volatile("" : "+v"(own));
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint32_t at = at_rows[g * 16 + (own & 15)];
    vec8 row[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const uint32_t piece = (uint32_t)(kb * 64 + (own >> 4) * 16);
      row[kb] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(
                                             a_rows, piece < (uint32_t)row_bytes ? at + piece : kNoRow, 0, 0));
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float4v product = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        product = E::mfma(*reinterpret_cast<const vec8 *>(filter + (nb * KB + kb) * 1024 + own * 16), row[kb], product);
      if (at != kNoRow) acc[g][nb] += product;  // (a lane's results are of its own row)
      asm volatile("" ::: "memory");            // one block's fragments in registers at a time
    }
  }
}

// The filled slots of all threads, for the collision check; by the whole workgroup, behind its last use of the map.
__device__ __forceinline__ void storeDenseSlots(DenseMap &map, int slots, int32_t *filled) {
  __syncthreads();
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) slots += __shfl_xor(slots, d, kWave);
  if ((threadIdx.x & 63) == 0) map.count[threadIdx.x >> 6] = slots;
  __syncthreads();
  if (threadIdx.x == 0) {
    int all = 0;
    for (int w = 0; w < kDenseThreads / 64; ++w) all += map.count[w];
    filled[blockIdx.x] = all;
  }
}

// ---- rows of up to 64 bytes
//
// Operand-order loads take each such row whole, so rows come straight into the operand registers (lane (row,
// quarter) loads 16 bytes) and whole phases of two offsets are in flight; nothing is skipped: a group
// without rows multiplies zeros.  A wave owns two row groups and ALL result columns.
// Filter.  The waves share an offset's filter: its fragments travel from global memory into a
// ring of two LDS buffers, a phase of two offsets at a time, and every wave reads all of
// them from there, once per offset for both its row groups.  One barrier per phase hands a
// buffer over; it waits for LDS traffic only, and each wave waits for its own requests itself
// (__syncthreads() would make every wave wait for all loads in flight).
// What bounds it is the loop itself (16 channels, 80 k rows, 27 offsets, half the slots filled: 37 us).  Rows through
// LDS as below are no faster here (248 636 rows of a scene, with the filter's packing: 16 -> 16 38 us against 46,
// 32 -> 32 47 against 47).
// Workgroups a CU: sums of two row groups and eight column blocks take the registers of two.
constexpr int densePerCu(int C) { return C >= 128 ? 2 : 4; }

template <typename E, int Q, int C, typename SRC>
__global__ __launch_bounds__(kDenseThreads)
    __attribute__((amdgpu_waves_per_eu(densePerCu(C), densePerCu(C))))
void gatherConvDense(const typename E::storage *A, uint32_t a_size, ConvRows conv,
                     const typename E::storage *packedW, SRC source, int R, int K,
                     typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int WAVES = kDenseThreads / 64;
  constexpr int G = kDenseGroups / WAVES;
  constexpr int NB = C / 16;                 // 16-column blocks, all of them in every wave
  constexpr int KC = kDenseChunk;
  constexpr int FRAGS = NB;                  // 1 KiB filter fragments per offset
  constexpr int W_BYTES = FRAGS * 1024;
  constexpr int OPP = 2;                     // offsets per phase
  constexpr int BUF_FRAGS = OPP * FRAGS;
  constexpr int FPW = (BUF_FRAGS + WAVES - 1) / WAVES;
  static_assert(Q <= E::kChunk, "one fragment a row");

  __shared__ __attribute__((aligned(1024))) char s_w[2 * BUF_FRAGS * 1024];
  __shared__ __attribute__((aligned(16))) DenseMap s_map;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_per_xcd = gridDim.x >> 3;  // neighbouring tiles on one XCD, as above
  const int tile = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  const int r0 = tile * kDenseRows;
  if constexpr (!SRC::kSegments) {
    if (notWanted(source.run_if)) return;
  }
  if (r0 >= R) {
    if constexpr (!SRC::kSegments) {
      if (tid == 0) source.filled[blockIdx.x] = 0;
    }
    return;
  }
  if constexpr (SRC::kSegments) {
    if (*source.verdict == source.ticket) {
      if (!source.leave_if_unordered) denseTileOutOfOrder<E>(s_map, A, conv, source, r0, R, K, result);
      return;
    }
  }
  const int pair = lane & 15;
  const int quad = lane >> 4;
  const __amdgpu_buffer_rsrc_t a_rows = rowsBuffer(A, a_size);
  const char *w_base = reinterpret_cast<const char *>(packedW) + lane * 16;
  const unsigned long long *const nonfinite =
      reinterpret_cast<const unsigned long long *>(reinterpret_cast<const char *>(packedW) + (size_t)K * W_BYTES);
  const uint32_t w_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)s_w;
  const int row_first = wave * (G * 16) + pair;  // this lane's row in its wave's first group
  // a lane's quarter of a row; behind the row's own bytes: nowhere (zeros)
  const uint32_t piece_at = quad * 16 < conv.row_bytes ? (uint32_t)quad * 16u : kNoRow;

  float4v acc[G][NB];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
  int slots = 0;  // filled map slots this thread staged

  for (int kc = 0; kc < K; kc += KC) {
    const int kn = (K - kc) < KC ? (K - kc) : KC;
    __syncthreads();  // the chunk before is finished with s_map and the filter buffers
    slots += fillDenseMap(s_map, source, nonfinite, conv.row_bytes, tile, r0, R, kc, kn, K);
    const bool has = lane < kn && s_map.groups[lane < kn ? lane : 0] != 0;
    const bool finite = s_map.finite[lane < kn ? lane : 0] != 0;
    // offsets of the chunk that have a pair in this tile; those of them whose filter is not finite go by themselves
    const uint32_t offsets = (uint32_t)__ballot(has && finite);
    for (uint32_t left = (uint32_t)__ballot(has && !finite); left != 0; left &= left - 1) {
      const int kk = __builtin_ctz(left);
      addOffsetApart<E, G, NB, 1>(acc, a_rows, &s_map.at[kk][wave * (G * 16)],
                                  reinterpret_cast<const char *>(packedW) + (size_t)(kc + kk) * W_BYTES, conv.row_bytes);
    }
    if (offsets == 0) continue;
    // A phase: the OPP lowest offsets of `left` (fewer at the end), which are taken out of it.
    auto next_phase = [](uint32_t &left) -> uint32_t {
      uint32_t rest = left;
#pragma unroll
      for (int o = 0; o < OPP; ++o) rest &= rest - 1;
      const uint32_t phase = left & ~rest;
      left = rest;
      return phase;
    };
    // Fragment f of a phase's filters (its offsets in ascending order), as bytes of the packed
    // filter.  Behind the phase's last offset: fragments of another offset of the walk, which are
    // multiplied by zeros if at all.
    auto fragment_of = [&](uint32_t phase, int f) -> const char * {
      uint32_t left = phase;
#pragma unroll
      for (int o = 1; o < OPP; ++o)
        if (f >= o * FRAGS && (left & (left - 1)) != 0) left &= left - 1;
      const int k = __builtin_ctz(left != 0 ? left : offsets);
      return w_base + ((size_t)(kc + k) * FRAGS + f % FRAGS) * 1024;
    };
    // The filters of a phase's offsets into half `half` of the ring: fragment f by wave f % WAVES.
    auto filters_to_lds = [&](uint32_t phase, int half) {
#pragma unroll
      for (int t = 0; t < FPW; ++t) {
        const int f = wave + t * WAVES;
        if (BUF_FRAGS % WAVES == 0 || f < BUF_FRAGS)
          requestToLds(fragment_of(phase, f), w_lds + (half * BUF_FRAGS + f) * 1024);
      }
    };
    // Rows in one of two sets of registers, filters in one of two ring buffers.
    vec8 rows_a[OPP][G], rows_b[OPP][G];
    auto request_phase = [&](uint32_t phase, int half, vec8 (&rows)[OPP][G]) {
      filters_to_lds(phase, half);
      uint32_t left = phase;
#pragma unroll
      for (int o = 0; o < OPP; ++o) {
        const uint32_t nowhere = left != 0 ? 0u : kNoRow;
        const int kk = left != 0 ? __builtin_ctz(left) : 0;
        left &= left - 1;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const uint32_t at = s_map.at[kk][row_first + g * 16] | nowhere;
          rows[o][g] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(
                                                    a_rows, __builtin_elementwise_add_sat(at, piece_at), 0, 0));
        }
      }
    };
    // Everything this wave has requested is there.  The rows pass through an empty statement
    // that the compiler must take for their last writer: it then places its own wait for their
    // loads here, and not in front of their first use, behind the next phase's requests, which
    // it would wait for as well.
    auto landed = [&](vec8 (&rows)[OPP][G]) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int o = 0; o < OPP; ++o)
#pragma unroll
        for (int g = 0; g < G; ++g) asm volatile("" : "+v"(rows[o][g]));
    };
    auto multiply_phase = [&](int half, const vec8 (&rows)[OPP][G]) {
      const char *filters = s_w + half * BUF_FRAGS * 1024 + lane * 16;
#pragma unroll
      for (int o = 0; o < OPP; ++o)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const vec8 w = *reinterpret_cast<const vec8 *>(filters + o * W_BYTES + nb * 1024);
#pragma unroll
          for (int g = 0; g < G; ++g) acc[g][nb] = E::mfma(w, rows[o][g], acc[g][nb]);
        }
    };
    // The rows' last values are done with.  (Requests behind a branch else leave the compiler a choice of old and new rows:
    // it copied the next phase's, and so waited for them in front of this phase's multiplies.  us of this kernel, half a
    // scene's rows, 0.25 filled, without / with this: 120 000 rows fp16 32 -> 64 36/25, fp32 16 -> 16 29.0/27.6; 3 000 rows
    // 19.5/16.0, 16.6/14.2.)
    auto forget = [&](vec8 (&rows)[OPP][G]) {
#pragma unroll
      for (int o = 0; o < OPP; ++o)
#pragma unroll
        for (int g = 0; g < G; ++g) asm volatile("" : "=v"(rows[o][g]));
    };
    uint32_t left = offsets;
    uint32_t phase = next_phase(left);
    request_phase(phase, 0, rows_a);
    landed(rows_a);
    ldsBarrier();
    while (true) {
      phase = next_phase(left);
      forget(rows_b);
      if (phase != 0) request_phase(phase, 1, rows_b);
      multiply_phase(0, rows_a);
      if (phase == 0) break;
      landed(rows_b);
      ldsBarrier();
      phase = next_phase(left);
      forget(rows_a);
      if (phase != 0) request_phase(phase, 0, rows_a);
      multiply_phase(1, rows_b);
      if (phase == 0) break;
      landed(rows_a);
      ldsBarrier();
    }
  }
  // lane holds result columns 16*nb + 4*quad + (0..3) of row 16*g + pair of its wave's rows
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int r = r0 + row_first + g * 16;
    if (r >= R) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      S tmp[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) E::store(&tmp[e], activated(acc[g][nb][e], conv.relu));
      storeColumns<E>(result + (size_t)r * conv.c, nb * 16 + quad * 4, conv.c, tmp);
    }
  }
  if constexpr (!SRC::kSegments) storeDenseSlots(s_map, slots, source.filled);
}

// ---- rows above 64 bytes
//
// The waves of a workgroup split the result COLUMNS between them (below 64 columns the rows as well) and share the
// tile's gathered rows: a phase's rows go from memory straight into one of two LDS buffers (16-byte loads in the
// order of the rows, four or eight rows a load; their pieces permuted so that operand reads meet no bank
// twice), while the phase before is multiplied, and every wave reads them from there.  A wave's filter
// columns are its own: they come into registers, one phase ahead as well.  Row groups without a partner at
// an offset are neither loaded nor multiplied.  Rows of 256 bytes take two phases an offset, half of their
// channels each, so that three workgroups share a CU; what one of them waits for the others multiply through.
//
// What bounds it: no unit by itself, but a phase's round trip.  128 -> 128 of the scene below, by counters: the way of loaded
// data into a CU is busy 62 % of the time, with 27 bytes a clock for rows (20 KB an offset and tile, 0.6 of the groups
// present) and filters (32 KB), the matrix cores 29 %, VALU issue 18 %; a wave waits 42 % of its life for loads or at a
// barrier and 35 % for its turn to issue.  Loads in operand order, 16 rows
// of 64 bytes each, take the address unit 64 clocks a KiB, whole rows 20, which is why rows go through LDS.  us,
// 248 636 rows of a scene, 27 offsets, with the filter's packing, this kernel / filters through LDS with
// rows in operand order (128) or through registers and LDS (64):
//   fp16 128 -> 128 167/210    64 -> 64 82/95
// Of two offsets a phase (64 channels: 93), tiles of 256 rows (128: 233; 64: 123), whole rows of 256 bytes (185),
// quarters (181) and 32 columns a wave at 64 (86) none is faster.
// A phase of two pieces (DEPTH) is for few tiles and for rows in no order: denseDepth.
// OFFSETS: an offset's product is a chain of its own, added to the row's sum when it is whole, as the pair-list kernels
// add: their bits (128 -> 128 takes the registers of two workgroups a CU for it; useDenseKernel has both sides' times).
struct StagedPlan {
  int column_waves;   // waves side by side; the others are below each other
  int column_blocks;  // of 16 result columns, of a wave
  int parts;          // phases a row's channels are split over
};
constexpr StagedPlan stagedPlan(int elem_bytes, int Q, int C) {
  return StagedPlan{C >= 64 ? 4 : (C >= 32 ? 2 : 1), C >= 128 ? 2 : 1, Q * elem_bytes >= 256 ? 2 : 1};
}
// Workgroups a CU.
constexpr int stagedPerCu(int Q, int C, bool offsets, int depth) {
  return depth == 2 || (offsets && Q == 128 && C == 128) ? 2 : 3;
}
// Where piece `piece` of a staged row lies among its row's pieces: at piece ^ this.
__device__ __forceinline__ int stagedSwizzle(int row) {
  return (row >> 1) & 7;
}

// 16 bytes per lane from byte `offset` of a buffer straight into LDS (as requestToLds); zeros for offsets behind its
// end.
__device__ __forceinline__ void requestRowsToLds(u32x4 rows, uint32_t offset, uint32_t lds_address) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds_address), "v"(offset), "s"(rows) : "memory", "m0");
}

// The same with 4 bytes per lane.
__device__ __forceinline__ void requestWordsToLds(u32x4 words, uint32_t offset, uint32_t lds_address) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :: "s"(lds_address), "v"(offset), "s"(words) : "memory", "m0");
}

template <typename E, int Q, int C, bool OFFSETS, int DEPTH, typename SRC>
__global__ __launch_bounds__(kDenseThreads)
    __attribute__((amdgpu_waves_per_eu(stagedPerCu(Q, C, OFFSETS, DEPTH), stagedPerCu(Q, C, OFFSETS, DEPTH))))
void gatherConvDenseStaged(const typename E::storage *A, uint32_t a_size, ConvRows conv,
                           const typename E::storage *packedW, SRC source, int R, int K, typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr StagedPlan PLAN = stagedPlan((int)sizeof(S), Q, C);
  constexpr int WAVES = kDenseThreads / 64;
  constexpr int CW = PLAN.column_waves;
  constexpr int NB = PLAN.column_blocks;         // of this wave
  constexpr int G = kDenseGroups / (WAVES / CW);  // row groups of this wave
  constexpr int KC = kDenseChunk;
  constexpr int RB = Q * (int)sizeof(S);
  constexpr int PARTS = PLAN.parts;
  constexpr int SB = RB / PARTS;                 // bytes of a row staged in one phase
  constexpr int KB = RB / 64;                    // fragments of a row
  constexpr int KP = KB / PARTS;
  constexpr int PPR = SB / 16;
  constexpr int RPL = 1024 / SB;                 // rows a load of 1 KiB stages
  constexpr int LPG = 16 / RPL;                  // loads a row group
  constexpr int GPW = kDenseGroups / WAVES;      // row groups a wave stages
  constexpr int BUFFER = kDenseRows * SB;
  constexpr int W_BYTES = (C / 16) * KB * 1024;  // packed filter of an offset
  static_assert(SB == 128 && CW * NB * 16 == C && WAVES % CW == 0, "split");

  __shared__ __attribute__((aligned(1024))) char s_rows[2 * DEPTH * BUFFER];
  __shared__ __attribute__((aligned(16))) DenseMap s_map;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_per_xcd = gridDim.x >> 3;  // neighbouring tiles on one XCD, as above
  const int tile = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  const int r0 = tile * kDenseRows;
  if constexpr (!SRC::kSegments) {
    if (notWanted(source.run_if)) return;
  }
  if (r0 >= R) {
    if constexpr (!SRC::kSegments) {
      if (tid == 0) source.filled[blockIdx.x] = 0;
    }
    return;
  }
  if constexpr (SRC::kSegments) {
    if (*source.verdict == source.ticket) {
      if (!source.leave_if_unordered) denseTileOutOfOrder<E>(s_map, A, conv, source, r0, R, K, result);
      return;
    }
  }
  const int pair = lane & 15;
  const int quad = lane >> 4;
  const int first_group = wave / CW * G;          // this wave's rows,
  const int first_block = wave % CW * NB;         // and columns
  const int row_first = first_group * 16 + pair;  // this lane's row in the first group
  const char *const w_base = reinterpret_cast<const char *>(packedW) + first_block * KB * 1024 + lane * 16;
  const unsigned long long *const nonfinite =
      reinterpret_cast<const unsigned long long *>(reinterpret_cast<const char *>(packedW) + (size_t)K * W_BYTES);
  const uint32_t rows_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)s_rows;
  // Where this lane's operand pieces of its wave's first row group lie.
  const char *lane_rows[KP];
#pragma unroll
  for (int kb = 0; kb < KP; ++kb) lane_rows[kb] = s_rows + row_first * SB + ((kb * 4 + quad) ^ stagedSwizzle(pair)) * 16;
  // Which piece of a row this lane stages, by load of a group.
  const __amdgpu_buffer_rsrc_t a_rows = rowsBuffer(A, a_size);
  const u32x4 rows_words = {(uint32_t)reinterpret_cast<uintptr_t>(A), (uint32_t)(reinterpret_cast<uintptr_t>(A) >> 32),
                            a_size, 0x00020000u};  // (a_rows, as requestRowsToLds takes it)
  uint32_t piece_of[PARTS][LPG];
#pragma unroll
  for (int part = 0; part < PARTS; ++part)
#pragma unroll
    for (int j = 0; j < LPG; ++j) {
      const uint32_t piece = (uint32_t)((lane % PPR) ^ stagedSwizzle(j * RPL + lane / PPR)) * 16u + part * SB;
      piece_of[part][j] = piece < (uint32_t)conv.row_bytes ? piece : kNoRow;
    }

  float4v acc[G][NB];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[g][nb] = float4v{0.f, 0.f, 0.f, 0.f};
  float4v held[OFFSETS && PARTS > 1 ? G : 1][OFFSETS && PARTS > 1 ? NB : 1];  // an offset's product, of its first part
  int slots = 0;  // filled map slots this thread staged

  for (int kc = 0; kc < K; kc += KC) {
    const int kn = (K - kc) < KC ? (K - kc) : KC;
    __syncthreads();  // the chunk before is finished with s_map and the row buffers
    slots += fillDenseMap(s_map, source, nonfinite, conv.row_bytes, tile, r0, R, kc, kn, K);
    const int lane_groups = lane < kn ? (int)s_map.groups[lane] : 0;
    const bool lane_finite = s_map.finite[lane < kn ? lane : 0] != 0;
    // offsets of the chunk that have a pair in this tile; those of them whose filter is not finite go by themselves
    const uint32_t offsets = (uint32_t)__ballot(lane_groups != 0 && lane_finite);
    for (uint32_t left = (uint32_t)__ballot(lane_groups != 0 && !lane_finite); left != 0; left &= left - 1) {
      const int kk = __builtin_ctz(left);
      addOffsetApart<E, G, NB, KB>(
          acc, a_rows, &s_map.at[kk][first_group * 16],
          reinterpret_cast<const char *>(packedW) + (size_t)(kc + kk) * W_BYTES + first_block * KB * 1024, conv.row_bytes);
    }
    if (offsets == 0) continue;
    // A piece is a part of one offset's channels, a phase DEPTH pieces.  kk < 0: no offset is left; nothing is staged and
    // nothing multiplied.
    uint32_t left = offsets;
    auto next_offset = [&]() -> int {
      const int kk = left != 0 ? __builtin_ctz(left) : -1;
      left &= left - 1;
      return kk;
    };
    auto groups_of = [&](int kk) -> uint32_t {
      return kk < 0 ? 0u : (uint32_t)__builtin_amdgcn_readlane(lane_groups, kk);
    };
    typedef vec8 Filters[NB][KP];
    // The row groups the wave stages straight into LDS, and its filter columns into registers.
    auto request = [&](int kk, int part, int buffer, Filters &w) {
      const int there = kk < 0 ? 0 : kk;
      uint32_t at[GPW][LPG];  // (all places in the map are read before the first address is formed)
#pragma unroll
      for (int t = 0; t < GPW; ++t)
#pragma unroll
        for (int j = 0; j < LPG; ++j) at[t][j] = s_map.at[there][(wave + t * WAVES) * 16 + j * RPL + lane / PPR];
      const char *const filter = w_base + (size_t)(kc + there) * W_BYTES;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int kb = 0; kb < KP; ++kb)
          w[nb][kb] = *reinterpret_cast<const vec8 *>(filter + (nb * KB + part * KP + kb) * 1024);
#pragma unroll
      for (int t = 0; t < GPW; ++t)
#pragma unroll
        for (int j = 0; j < LPG; ++j) {
          at[t][j] = __builtin_elementwise_add_sat(at[t][j], piece_of[part][j]);
          asm volatile("" : "+v"(at[t][j]));
        }
      const uint32_t groups = groups_of(kk) >> wave;
#pragma unroll
      for (int t = 0; t < GPW; ++t) {
        if ((groups >> (t * WAVES) & 1u) == 0) continue;
#pragma unroll
        for (int j = 0; j < LPG; ++j)
          requestRowsToLds(rows_words, at[t][j],
                           rows_lds + (uint32_t)(buffer * BUFFER + ((wave + t * WAVES) * LPG + j) * 1024));
      }
    };
    // Piece `first` + j of the trip's 2 * DEPTH, each with a buffer of its own; `before`: the offset of the piece in front.
    auto request_phase = [&](auto first, int before, int (&of)[DEPTH], Filters (&w)[DEPTH]) {
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) {
        of[j] = (first + j) % PARTS == 0 ? next_offset() : (j > 0 ? of[j - 1] : before);
        request(of[j], (first + j) % PARTS, first + j, w[j]);
      }
    };
    // Everything this wave has requested is there.  The filters pass through an empty statement that the
    // compiler must take for their last writer: its own wait for their loads then lies here, and not in front
    // of their first use, behind the next phase's requests, which it would wait for as well.
    auto landed = [&](Filters (&w)[DEPTH]) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < DEPTH; ++j)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int kb = 0; kb < KP; ++kb) asm volatile("" : "+v"(w[j][nb][kb]));
    };
    // (a group's rows are read while the group before is multiplied; those of a group without partners are what
    // the buffer held before, and nobody multiplies them)
    auto multiply = [&](int kk, int part, int buffer, const Filters &w) {
      const uint32_t groups = groups_of(kk) >> first_group;
      vec8 row[2][KP];
      auto read_group = [&](int g) {
#pragma unroll
        for (int kb = 0; kb < KP; ++kb)
          row[g & 1][kb] = *reinterpret_cast<const vec8 *>(lane_rows[kb] + buffer * BUFFER + g * 16 * SB);
      };
      read_group(0);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (g + 1 < G) read_group(g + 1);
        __builtin_amdgcn_sched_barrier(0);
        if ((groups >> g & 1u) == 0) continue;
        if constexpr (OFFSETS) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            float4v product = part > 0 ? held[g][nb] : float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KP; ++kb) product = E::mfma(w[nb][kb], row[g & 1][kb], product);
            if (part == PARTS - 1) acc[g][nb] += product;
            else held[g][nb] = product;
          }
        } else {
#pragma unroll
          for (int kb = 0; kb < KP; ++kb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[g][nb] = E::mfma(w[nb][kb], row[g & 1][kb], acc[g][nb]);
        }
      }
    };
    // (two phases a trip and one way out of the loop, at the price of an empty phase at the end of an
    // odd number of them: with a second way out the compiler waits for all loads in front of every use)
    auto multiply_phase = [&](auto first, const int (&of)[DEPTH], const Filters (&w)[DEPTH]) {
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) multiply(of[j], (first + j) % PARTS, first + j, w[j]);
    };
    constexpr std::integral_constant<int, 0> kEven{};
    constexpr std::integral_constant<int, DEPTH> kOdd{};
    Filters w_a[DEPTH], w_b[DEPTH];
    int now[DEPTH], after[DEPTH];
    request_phase(kEven, -1, now, w_a);
    landed(w_a);
    ldsBarrier();
    do {
      request_phase(kOdd, now[DEPTH - 1], after, w_b);
      multiply_phase(kEven, now, w_a);
      landed(w_b);
      ldsBarrier();
      request_phase(kEven, -1, now, w_a);
      multiply_phase(kOdd, after, w_b);
      landed(w_a);
      ldsBarrier();
    } while (now[0] >= 0);
  }
  // lane holds result columns 16*nb + 4*quad + (0..3) of row 16*g + pair of its wave's rows
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int r = r0 + row_first + g * 16;
    if (r >= R) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      S tmp[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) E::store(&tmp[e], activated(acc[g][nb][e], conv.relu));
      storeColumns<E>(result + (size_t)r * conv.c, (first_block + nb) * 16 + quad * 4, conv.c, tmp);
    }
  }
  if constexpr (!SRC::kSegments) storeDenseSlots(s_map, slots, source.filled);
}

// ---- result rows in one pair each -------------------------------------------------------
//
// Where no result row is in two pairs (the input rows of a 2x2x2 layer with stride 2, for its input's gradient and for
// the inverse layer) there is nothing to add up: a workgroup multiplies `singlePairs` pairs of ONE offset, whatever
// rows they belong to, and stores the products.  Its blocks are full, its filter is one, and it needs no sums in
// LDS and no cut table.  The waves split columns and rows as in the dense kernel above; rows go straight into LDS.
// What bounds it is the chain of three dependent loads (pairs, rows, results) of workgroups that live for 5 us, and
// memory; in fp32 the multiplies, of which those behind a row's end are left out (39 -> 35 us with 96 channels in tiles of
// 128).  us of the gather kernel alone, 2x2x2 stride 2, the list kernels / this one: fp32 96 -> 64 of 200 000 rows
// 76/35, bf16 128 -> 96 of 100 000 31/16, fp16 128 -> 64 of 150 000 24/15, 64 -> 64 of 100 000 15/10, 32 -> 16 9.8/5.8.
constexpr int singlePairs(int row_bytes) { return row_bytes >= 512 ? 64 : 128; }
constexpr int singlePieceAt(int row_bytes, int row, int piece) {
  if (row_bytes >= 256) return piece ^ (row & 15);
  if (row_bytes == 128) return piece ^ (row >> 1 & 7);
  const int r = row >> 2 & 3;  // 0 2 3 1: the 16 rows whose pieces are read together meet all banks
  return piece ^ (r << 1 & 2) ^ (r >> 1 & 1) * 3;
}

template <typename E, int Q, int C>
__global__ __launch_bounds__(kDenseThreads) void gatherConvSingle(
    const typename E::storage *A, uint32_t a_size, ConvRows conv, const typename E::storage *packedW,
    const int32_t *__restrict__ pairs, int L, int row_col, int src_col, OffsetCounts counts, OffsetBlocks blocks, int K,
    int R, int n_src, typename E::storage *result) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int WAVES = kDenseThreads / 64;
  constexpr int RB = Q * (int)sizeof(S) < 64 ? 64 : Q * (int)sizeof(S);
  constexpr int T = singlePairs(RB);
  constexpr int CW = stagedPlan((int)sizeof(S), Q, C).column_waves, NB = stagedPlan((int)sizeof(S), Q, C).column_blocks;
  constexpr int GROUPS = T / 16;
  constexpr int G = GROUPS / (WAVES / CW);
  constexpr int KB = RB / 64;
  constexpr int PPR = RB / 16;
  constexpr int RPL = 1024 / RB;  // rows a load of 1 KiB stages
  constexpr int LPG = 16 / RPL;
  __shared__ __attribute__((aligned(1024))) char s_rows[T * RB];
  __shared__ uint32_t s_src[T];  // where a pair's gathered row begins; kNoRow: the pair adds nothing
  __shared__ int s_row[T];       // its result row, or -1

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pair = lane & 15, quad = lane >> 4;
  int lo = 0, hi = K - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (blocks.first[mid] <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
  }
  const int k = lo, p0 = ((int)blockIdx.x - blocks.first[k]) * T;
  if (tid < T) {
    int row = -1, src = 0;
    if (p0 + tid < counts.n[k]) {
      const int32_t *const list = pairs + (size_t)k * 2 * L + p0 + tid;
      row = list[(size_t)row_col * L];
      src = list[(size_t)src_col * L];
    }
    s_src[tid] = (unsigned)src < (unsigned)n_src ? (uint32_t)src * (uint32_t)conv.row_bytes : kNoRow;
    s_row[tid] = (unsigned)row < (unsigned)R ? row : -1;
  }
  const int first_group = wave / CW * G, first_block = wave % CW * NB;
  const char *const filter =
      reinterpret_cast<const char *>(packedW) + (size_t)(k * (C / 16) + first_block) * KB * 1024 + lane * 16;
  vec8 w[NB][KB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) w[nb][kb] = *reinterpret_cast<const vec8 *>(filter + (nb * KB + kb) * 1024);
  ldsBarrier();
  const u32x4 rows_words = {(uint32_t)reinterpret_cast<uintptr_t>(A), (uint32_t)(reinterpret_cast<uintptr_t>(A) >> 32),
                            a_size, 0x00020000u};
  const uint32_t rows_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)s_rows;
#pragma unroll
  for (int t = 0; t < GROUPS / WAVES; ++t) {
    uint32_t at[LPG];
#pragma unroll
    for (int j = 0; j < LPG; ++j) {
      const int row = (wave + t * WAVES) * 16 + j * RPL + lane / PPR;
      // (the swizzle is its own inverse)
      const uint32_t piece = (uint32_t)singlePieceAt(RB, row & 15, lane % PPR) * 16u;
      at[j] = __builtin_elementwise_add_sat(s_src[row], piece < (uint32_t)conv.row_bytes ? piece : kNoRow);
    }
#pragma unroll
    for (int j = 0; j < LPG; ++j) asm volatile("" : "+v"(at[j]));
#pragma unroll
    for (int j = 0; j < LPG; ++j)
      requestRowsToLds(rows_words, at[j], rows_lds + (uint32_t)(((wave + t * WAVES) * LPG + j) * 1024));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  ldsBarrier();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int in_tile = (first_group + g) * 16 + pair;
    const char *const rows = s_rows + in_tile * RB;
    vec8 row[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      row[kb] = *reinterpret_cast<const vec8 *>(rows + singlePieceAt(RB, pair, kb * 4 + quad) * 16);
    const int to = s_row[in_tile];
    const bool adds = s_src[in_tile] != kNoRow;  // (a row of zeros times a filter that is not finite is not zero)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float4v product = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        if (kb * 64 < conv.row_bytes) product = E::mfma(w[nb][kb], row[kb], product);
      if (to < 0) continue;
      // (a sum that starts from zero, as in the other kernels: a product of -0 is stored as 0)
      S tmp[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) E::store(&tmp[e], activated(adds ? 0.f + product[e] : 0.f, conv.relu));
      storeColumns<E>(result + (size_t)to * conv.c, (first_block + nb) * 16 + quad * 4, conv.c, tmp);
    }
  }
}

// ---- pairs that lost their map slot -----------------------------------------------
// Runs behind every gather kernel and returns at once when the kernels found as many
// filled map slots as there are pairs inside their tensors (always, for a rulebook built
// from distinct coordinates).  Otherwise some pairs of one offset share a result row:
// every pair is looked up again, the first one that finds its partner in the slot claims
// it (the kernels have multiplied that one), and each of the others is added to its
// result row here.  The result rows are split into windows of kRepairPoolRows rows; a
// workgroup takes every gridDim.x-th window, reads all pairs and keeps those of its
// window, so no two workgroups touch the same row, map slot or shadow entry.  A touched
// row is rebuilt in the workgroup's fp32 pool (indexed through `shadow`): first the
// partners its map slots hold, as the kernel summed them, then the lost pairs as the
// scan meets them, and it is rounded into the result once, the same single rounding as
// any other row.  Which of the colliding pairs owned the slot depends on the order their
// stores landed in, so the last bits of such rows can differ from run to run; rows
// without collisions are not touched.
constexpr int kRepairPoolRows = 2048;
constexpr int kRepairBlocks = 32;

struct RepairScratch {
  int32_t *shadow;    // [R] pool row of a result row, or -1
  int32_t *pool_row;  // [kRepairBlocks, kRepairPoolRows] result row of a pool row
  float *pool;        // [kRepairBlocks, kRepairPoolRows, C]
};

template <typename E>
__global__ __launch_bounds__(256) void repairLostPairs(
    const typename E::storage *A, int Q, const typename E::storage *W, int64_t sK, int64_t sQ,
    int64_t sC, const int32_t *pairs, int L, int row_col, int src_col, int R, int n_src, int K,
    int row_base, OffsetCounts inl, const int32_t *dev_counts, int32_t *map,
    const int32_t *filled, int n_filled, const int32_t *accepted, int n_accepted, int C,
    RepairScratch scratch, bool relu, typename E::storage *result, RunIf run_if) {
  if (notWanted(run_if)) return;
  __shared__ int s_found;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (tid == 0) s_found = 0;
  __syncthreads();
  // filled slots the gather kernel met, less the pairs the scatter put into the map
  int mine = 0;
  for (int i = tid; i < n_filled; i += 256) mine += filled[i];
  for (int i = tid; i < n_accepted; i += 256) mine -= accepted[i];
  mine = waveInclusiveScan(mine);
  if (lane == 63 && mine != 0) atomicAdd(&s_found, mine);
  __syncthreads();
  if (s_found == 0) return;

  __shared__ int s_row[256];
  __shared__ int s_src[256];
  __shared__ int s_wave_lost[4];
  __shared__ int s_pooled;  // pool rows in use
  int32_t *pool_row = scratch.pool_row + (size_t)blockIdx.x * kRepairPoolRows;
  float *pool = scratch.pool + (size_t)blockIdx.x * kRepairPoolRows * C;
  // Products of gathered rows with filter slices, summed into pool row `at`: below 256
  // result columns the workgroup is 256 / C groups of C threads, a group takes every
  // groups-th reduction channel and the groups' sums meet in shared memory, in group order.
  __shared__ float s_part[256];
  const int groups = C < 256 ? 256 / C : 1;
  const int g = C < 256 ? tid / C : 0;  // == groups: a thread without a part
  const int c_first = C < 256 ? tid % C : tid;
  // whole_row: every partner the map holds for result row `row` (claimed slots hold
  // -2 - partner), stored; else gathered row `row` times slice `k_one`, added.
  auto addProducts = [&](int at, int row, bool whole_row, int k_one) {
    for (int c = c_first; c < C; c += 256) {
      float part = 0.f;
      if (g < groups) {
        for (int kk = whole_row ? 0 : k_one; kk < (whole_row ? K : k_one + 1); ++kk) {
          int from = row;
          if (whole_row) {
            const int m = map[(size_t)kk * R + row];
            if (m == -1) continue;
            from = m >= 0 ? m : -2 - m;
          }
          const typename E::storage *a = A + (size_t)from * Q;
          const typename E::storage *w = W + (size_t)kk * sK + (size_t)c * sC;
          for (int q = g; q < Q; q += groups) part += E::load(a + q) * E::load(w + (size_t)q * sQ);
        }
      }
      if (groups > 1) {
        s_part[tid] = part;
        __syncthreads();
        if (g == 0) {
          part = 0.f;
          for (int gg = 0; gg < groups; ++gg) part += s_part[gg * C + c];
        }
      }
      if (g == 0) pool[(size_t)at * C + c] = whole_row ? part : pool[(size_t)at * C + c] + part;
      if (groups > 1) __syncthreads();
    }
  };
  const int n_windows = (R + kRepairPoolRows - 1) / kRepairPoolRows;
  for (int window = blockIdx.x; window < n_windows; window += gridDim.x) {
    const int r_lo = window * kRepairPoolRows;
    const int r_hi = r_lo + kRepairPoolRows < R ? r_lo + kRepairPoolRows : R;
    for (int i = r_lo + tid; i < r_hi; i += 256) scratch.shadow[i] = -1;
    if (tid == 0) s_pooled = 0;
    __syncthreads();
    for (int k = 0; k < K; ++k) {
      const int n = offsetCount(inl, dev_counts, k);
      const int32_t *base = pairs + (size_t)k * 2 * L;
      for (int p0 = 0; p0 < n; p0 += 256) {
        const int p = p0 + tid;
        int r = -1, src = -1;
        bool lost = false;
        if (p < n) {
          r = base[(size_t)row_col * L + p] - row_base;
          if (r >= r_lo && r < r_hi) {
            src = base[(size_t)src_col * L + p];
            if ((unsigned)src < (unsigned)n_src) {
              int32_t *slot = map + (size_t)k * R + r;
              // the claimed slot holds -2 - partner: no pair finds itself there twice
              lost = !(*slot == src && atomicCAS(slot, src, -2 - src) == src);
            }
          }
        }
        // most steps hold no pair of this window at all
        if (!__syncthreads_or(lost)) continue;
        // lost pairs of this step in pair order
        const unsigned long long b = __ballot(lost);
        if (lane == 0) s_wave_lost[wave] = __popcll(b);
        __syncthreads();
        int before = 0, total = 0;
        for (int w = 0; w < 4; ++w) {
          if (w < wave) before += s_wave_lost[w];
          total += s_wave_lost[w];
        }
        if (lost) {
          const int at = before + __popcll(b & ((1ull << lane) - 1ull));
          s_row[at] = r;
          s_src[at] = src;
        }
        __syncthreads();
        for (int i = 0; i < total; ++i) {
          const int row = s_row[i];
          int at = scratch.shadow[row];
          if (at < 0) {
            at = s_pooled;
            __syncthreads();  // everybody has read the pool's fill state
            if (tid == 0) {
              scratch.shadow[row] = at;
              pool_row[at] = row;
              s_pooled = at + 1;
            }
            // what the gather kernel summed: the partner every slot of the row holds
            addProducts(at, row, true, 0);
          }
          addProducts(at, s_src[i], false, k);
          __syncthreads();  // shadow and the pool row are in place for the next pair
        }
      }
    }
    // round the rebuilt rows into the result; the pool is free for the next window
    const int pooled = s_pooled;
    for (int i = 0; i < pooled; ++i) {
      const int r = pool_row[i];
      for (int c = tid; c < C; c += 256) E::store(result + (size_t)r * C + c, activated(pool[(size_t)i * C + c], relu));
    }
    __syncthreads();
  }
}

// Number of map slots that hold a partner, added to *total (cleared beforehand).
__global__ __launch_bounds__(256) void countFilledSlots(const int32_t *map, size_t n, int32_t *total) {
  __shared__ int s_sum;
  if (threadIdx.x == 0) s_sum = 0;
  __syncthreads();
  int mine = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    mine += map[i] >= 0 ? 1 : 0;
  mine = waveInclusiveScan(mine);
  if ((threadIdx.x & 63) == 63) atomicAdd(&s_sum, mine);
  __syncthreads();
  if (threadIdx.x == 0 && s_sum != 0) atomicAdd(total, s_sum);
}

// ---- backward filter -------------------------------------------------------------
// Where dW(k, ci, co) goes in filters_grad (element strides).
struct GradLayout {
  int64_t stride_k, stride_ci, stride_co;
};
__device__ __forceinline__ size_t gradOffset(const GradLayout &g, int k, int ci, int co) {
  return (size_t)(k * g.stride_k + ci * g.stride_ci + co * g.stride_co);
}

// One block = 32 x 64 tile of dW[k] over a contiguous slice of the offset's pairs.
template <typename E>
__global__ __launch_bounds__(256) void backwardFilterSimt(const typename E::storage *X,
                                                          const typename E::storage *dY,
                                                          const int32_t *pairs, int L,
                                                          int x_col, int n_in, int n_out, int Ci,
                                                          int Co, OffsetCounts inl,
                                                          const int32_t *dev_counts, int splits,
                                                          float *partial, GradLayout lay,
                                                          typename E::storage *dW) {
  constexpr int TI = 32, TO = 64, PC = 32;
  __shared__ float Xs[PC][TI + 1];
  __shared__ float Ys[PC][TO];
  __shared__ int s_in[PC];
  __shared__ int s_out[PC];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int tiles_o = (Co + TO - 1) / TO;
  const int ci0 = (blockIdx.x / tiles_o) * TI;
  const int co0 = (blockIdx.x % tiles_o) * TO;
  const int k = blockIdx.y;
  const int s = blockIdx.z;
  const int K = gridDim.y;
  const int n = offsetCount(inl, dev_counts, k);
  int per = (n + splits - 1) / splits;
  per = (per + PC - 1) / PC * PC;
  const int p_begin = s * per;
  const int p_end = (p_begin + per) < n ? (p_begin + per) : n;
  const int32_t *in_col = pairs + ((size_t)k * 2 + x_col) * L;
  const int32_t *out_col = pairs + ((size_t)k * 2 + 1 - x_col) * L;
  float acc[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int p0 = p_begin; p0 < p_end; p0 += PC) {
    if (tid < PC) {
      const int p = p0 + tid;
      int i = -1, o = -1;
      if (p < p_end) {
        i = in_col[p];
        o = out_col[p];
        if ((unsigned)i >= (unsigned)n_in || (unsigned)o >= (unsigned)n_out) i = o = -1;
      }
      s_in[tid] = i;
      s_out[tid] = o;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PC * TI / 256; ++i) {
      const int e = tid + i * 256;
      const int p = e / TI, c = e % TI;
      const int row = s_in[p];
      Xs[p][c] = (row >= 0 && ci0 + c < Ci) ? E::load(X + (size_t)row * Ci + ci0 + c) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < PC * TO / 256; ++i) {
      const int e = tid + i * 256;
      const int p = e / TO, c = e % TO;
      const int row = s_out[p];
      Ys[p][c] = (row >= 0 && co0 + c < Co) ? E::load(dY + (size_t)row * Co + co0 + c) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int p = 0; p < PC; ++p) {
      const float a0 = Xs[p][ty * 2], a1 = Xs[p][ty * 2 + 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float b = Ys[p][tx * 4 + j];
        acc[0][j] += a0 * b;
        acc[1][j] += a1 * b;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ci = ci0 + ty * 2 + i;
    if (ci >= Ci) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = co0 + tx * 4 + j;
      if (co >= Co) continue;
      const size_t e = ((size_t)k * Ci + ci) * Co + co;
      if (splits == 1) {
        E::store(dW + gradOffset(lay, k, ci, co), acc[i][j]);
      } else {
        partial[(size_t)s * K * Ci * Co + e] = acc[i][j];
      }
    }
  }
}

// dW[e] = sum over splits, in split order, rounded once.
template <typename E>
__global__ __launch_bounds__(256) void reduceFilterPartials(const float *partial, size_t n,
                                                            int splits, int Ci, int Co,
                                                            GradLayout lay,
                                                            typename E::storage *dW) {
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
    float s = 0.f;
    for (int i = 0; i < splits; ++i) s += partial[(size_t)i * n + e];
    const int co = (int)(e % Co);
    const size_t kc = e / Co;
    E::store(dW + gradOffset(lay, (int)(kc / Ci), (int)(kc % Ci), co), s);
  }
}

// ---- MFMA backward filter ----------------------------------------------------------
// dW[k] = X_k^T . dY_k over the pairs of offset k.  The pairs of every offset
// are cut into slices of slice_len pairs; one workgroup multiplies one slice of
// one offset and writes a fp32 Ci x Co partial tile, sliceSum adds the tiles of an
// offset in slice order (no float atomics, the same bits on every run).
struct SliceTable {
  int n[kMaxInlineK];      // pairs of the offset
  int first[kMaxInlineK];  // partial tiles in front of the offset's first one
  int tiles[kMaxInlineK];  // partial tiles of the offset
};

constexpr int kFilterStepPairs = 64;     // pairs multiplied per barrier
constexpr int kFilterIndexChunk = 1024;  // pair indices resident in LDS at once
constexpr int kFilterMaxSlices = 1024;   // about four workgroups per CU
// Many offsets with short lists (5 x 5 x 5) are cut into fewer slices: every slice costs a
// Ci x Co fp32 tile written and summed again (config 5a, 125 offsets: 137 us at 768 slices,
// 149 at 1024; the 27-offset network layers: 183 -> 165 us at 128 channels, 89 -> 77 at 64).
constexpr int kFilterMaxSlicesManyOffsets = 768;
constexpr int kFilterFewOffsets = 32;
constexpr int kFilterWalkChunk = 256;  // pairs a walk takes at a time
constexpr int kFilterShares = 8;       // shares of every list: the XCDs

// The order in which the workgroups take the slices: by the share of its offset's list that
// lies in front of a slice, so that the workgroups running at one time are at about the same
// rows of the feature and gradient tensors in all offsets (the lists ascend by row), and a
// row fetched for one offset is still in the L2 cache when the others want it.  Entry j names
// the offset of the j-th slice in that order; it is that offset's s-th slice when s earlier
// entries name the same offset.  Workgroup b takes entry (b % 8) * (grid / 8) + b / 8:
// neighbouring entries on one XCD, behind one L2.
struct SliceOrder {
  uint8_t offset[kFilterMaxSlices + kMaxInlineK];
};

struct SlicePlace {
  int k, slice;
};

// For all threads of a workgroup (one barrier inside).  k < 0: no slice for this workgroup.
__device__ __forceinline__ SlicePlace sliceOfWorkgroup(const SliceOrder &order, int total) {
  __shared__ int s_place[2];
  const int per_xcd = gridDim.x >> 3;
  const int j = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
  if (threadIdx.x < 64) {
    int k = -1, earlier = 0;
    if (j < total) {
      k = order.offset[j];
      for (int i = threadIdx.x; i < j; i += 64) earlier += order.offset[i] == k;
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) earlier += __shfl_xor(earlier, d, kWave);
    if (threadIdx.x == 0) {
      s_place[0] = k;
      s_place[1] = earlier;
    }
  }
  __syncthreads();
  SlicePlace at;
  at.k = s_place[0];
  at.slice = s_place[1];
  return at;
}

struct FilterWalk {
  int k, share, walker;
};

// Walks: with many pairs slices are so long that the workgroups of an XCD are spread over far more rows than
// its L2 holds, and a row comes from memory again for most of its offsets (248 636 rows, 2.85 M pairs, 128 x 128
// channels: 704 MB for tensors of 127 MB, at the rate a copy reaches).  Every list is then cut into
// `shares` equal shares, share s walked by workgroups of XCD s % 8: an offset's `walkers` take its chunks of
// kFilterWalkChunk pairs in turn, so that all workgroups of the XCD go through the share's rows together.
// 163 -> 130 us there, 64 x 64 channels 74 -> 65, 32 x 32 53 -> 50.
// `order` names the offsets of one share's workgroups.
__device__ __forceinline__ FilterWalk walkOfWorkgroup(const SliceOrder &order, int per_share, int shares) {
  __shared__ int s_place[2];
  const int i = (int)blockIdx.x >> 3;
  const int entry = i % per_share;
  if (threadIdx.x < 64) {
    const int k = order.offset[entry];
    int earlier = 0;
    for (int j = threadIdx.x; j < entry; j += 64) earlier += order.offset[j] == k;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) earlier += __shfl_xor(earlier, d, kWave);
    if (threadIdx.x == 0) {
      s_place[0] = k;
      s_place[1] = earlier;
    }
  }
  __syncthreads();
  return FilterWalk{s_place[0], (i / per_share) * 8 + ((int)blockIdx.x & 7), s_place[1]};
}

// The pairs of a workgroup: pair t of `length` (whole steps of kFilterStepPairs) at position at(t) of the
// offset's list, if that lies in front of `end`.
struct FilterRun {
  int k;     // -1: nothing to do
  int tile;  // partial tile the products go to
  int begin, end, stride, length;
  __device__ __forceinline__ int at(int t) const {
    return begin + t / kFilterWalkChunk * stride + t % kFilterWalkChunk;
  }
};

__device__ __forceinline__ FilterRun runOfWorkgroup(const SliceTable &tab, const SliceOrder &order, int entries,
                                                    int slice_len, int shares) {
  FilterRun run;
  if (shares > 0) {
    const FilterWalk walk = walkOfWorkgroup(order, entries, shares);
    const int n = tab.n[walk.k], walkers = tab.tiles[walk.k] / shares;
    run.k = walk.k;
    run.tile = tab.first[walk.k] + walk.share * walkers + walk.walker;
    run.begin = (int)((long long)n * walk.share / shares) + walk.walker * kFilterWalkChunk;
    run.end = (int)((long long)n * (walk.share + 1) / shares);
    run.stride = walkers * kFilterWalkChunk;
  } else {
    const SlicePlace at = sliceOfWorkgroup(order, entries);
    run.k = at.k;
    if (at.k < 0) return run;
    const int n = tab.n[at.k];
    run.tile = tab.first[at.k] + at.slice;
    run.begin = at.slice * slice_len;
    run.end = run.begin + slice_len < n ? run.begin + slice_len : n;
    run.stride = kFilterWalkChunk;
  }
  run.length = 0;  // (a walk behind the end of a short share still stores its tile, of zeros)
  if (run.begin < run.end) {
    const int before = (run.end - run.begin - 1) / run.stride;  // chunks in front of the last one
    const int last = run.end - (run.begin + before * run.stride);
    run.length = before * kFilterWalkChunk + ((last < kFilterWalkChunk ? last : kFilterWalkChunk) + kFilterStepPairs - 1) /
                                                 kFilterStepPairs * kFilterStepPairs;
  }
  return run;
}

// Both operands are needed with the pair index running along the MFMA's K
// dimension, i.e. transposed relative to the row-major tensors: rows are
// gathered with 16-byte loads and written to LDS transposed ([channel][pair],
// element-sized stores), from where an operand fragment (8 consecutive pairs of
// one channel, 4 for float) is one 16-byte read.  A wave stages 32 pairs x two
// neighbouring 16-byte pieces at a time: every transposed store of the wave then
// writes two runs of 32 consecutive pairs, which no two lanes share a bank in
// (with a row's pieces spread over eight lanes the same stores hit 8 banks and
// took 28 cycles each).  Wave w multiplies the 16-row blocks w, w+4, ... of dW[k]
// against all column blocks.  Rows are `rows.ci` and `rows.co` channels long: the channels
// behind them, up to CI and CO, are zeros.  WHOLE: rows of exactly CI and CO channels, with their
// lengths as constants (64 x 64 channels in fp32: 43 us, 46 with lengths from the arguments; the
// kernel behind this one, fp16: 64 x 64 14.6 against 15.2, 128 x 128 28.0 against 30.2).

// The channels of the feature and gradient rows, at most the CI and CO of the instance.
struct FilterGradRows {
  int ci, co;
};

// Elements [c0, c0 + 16 bytes) of a row of `channels`, zeros behind its end.  (Rows need no
// alignment: the memory path takes 16 bytes from any address.)
template <typename S>
__device__ __forceinline__ u32x4 rowPiece(const S *row, int c0, int channels) {
  constexpr int EPP = 16 / (int)sizeof(S);
  u32x4 piece = {0u, 0u, 0u, 0u};
  if (c0 + EPP <= channels) {
    __builtin_memcpy(&piece, row + c0, 16);
  } else {
#pragma unroll
    for (int e = 0; e < EPP; ++e) {
      if (c0 + e < channels) {
        if constexpr (sizeof(S) == 2)
          piece[e >> 1] |= (uint32_t)reinterpret_cast<const u16 *>(row)[c0 + e] << ((e & 1) * 16);
        else
          piece[e] = reinterpret_cast<const uint32_t *>(row)[c0 + e];
      }
    }
  }
  return piece;
}

template <typename E, int CI, int CO, bool WHOLE>
__global__ __launch_bounds__(256) void backwardFilterMfma(
    const typename E::storage *X, const typename E::storage *dY, FilterGradRows lengths, const int32_t *pairs, int L,
    int x_col, int n_in, int n_out, int K, SliceTable tab, SliceOrder order, int total_slices,
    int slice_len, int shares, float *partial) {
  typedef typename E::vec8 vec8;
  typedef typename E::storage S;
  constexpr int SP = kFilterStepPairs;
  constexpr int EPP = 16 / (int)sizeof(S);          // elements per 16-byte piece
  constexpr int STRIDE = SP * (int)sizeof(S) + 16;  // bytes per channel row: 16 rows hit 64 distinct banks
  constexpr int XP = SP * CI / EPP;                 // 16-byte pieces of X per step
  constexpr int YP = SP * CO / EPP;
  constexpr int XT = XP / 256 > 0 ? XP / 256 : 1;
  constexpr int YT = YP / 256 > 0 ? YP / 256 : 1;
  constexpr int XU = XP / 64;  // staging units (32 pairs x 2 pieces) of X per step
  constexpr int YU = YP / 64;
  const FilterGradRows rows = WHOLE ? FilterGradRows{CI, CO} : lengths;
  static_assert(SP == 64 && (CI / EPP) % 2 == 0 && (CO / EPP) % 2 == 0, "unit = 32 pairs x 2 pieces");
  constexpr int CBW = (CI / 16 + 3) / 4;  // row blocks per wave
  constexpr int COB = CO / 16;
  static_assert(XP % 256 == 0 || XP < 256, "piece split");
  static_assert(YP % 256 == 0 || YP < 256, "piece split");

  __shared__ __attribute__((aligned(16))) char s_x[CI * STRIDE];
  __shared__ __attribute__((aligned(16))) char s_y[CO * STRIDE];
  __shared__ int s_in[kFilterIndexChunk];
  __shared__ int s_out[kFilterIndexChunk];

  const FilterRun run = runOfWorkgroup(tab, order, total_slices, slice_len, shares);
  if (run.k < 0) return;
  const int k = run.k;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int32_t *in_col = pairs + ((size_t)k * 2 + x_col) * L;
  const int32_t *out_col = pairs + ((size_t)k * 2 + 1 - x_col) * L;

  float4v acc[CBW][COB];
#pragma unroll
  for (int a = 0; a < CBW; ++a)
#pragma unroll
    for (int b = 0; b < COB; ++b) acc[a][b] = float4v{0.f, 0.f, 0.f, 0.f};

  u32x4 xr[XT], yr[YT];
  auto fetch_step = [&](int local) {  // local = first pair of the step within the index chunk
#pragma unroll
    for (int i = 0; i < XT; ++i) {
      const int u = wave + i * 4;  // unit: pairs 32*(u&1).., pieces 2*(u>>1)..
      xr[i] = u32x4{0u, 0u, 0u, 0u};
      if (XU >= 4 || u < XU) {
        const int row = s_in[local + (u & 1) * 32 + (lane >> 1)];
        if (row >= 0)
          xr[i] = rowPiece(X + (size_t)row * rows.ci, ((u >> 1) * 2 + (lane & 1)) * EPP, rows.ci);
      }
    }
#pragma unroll
    for (int i = 0; i < YT; ++i) {
      const int u = wave + i * 4;
      yr[i] = u32x4{0u, 0u, 0u, 0u};
      if (YU >= 4 || u < YU) {
        const int row = s_out[local + (u & 1) * 32 + (lane >> 1)];
        if (row >= 0)
          yr[i] = rowPiece(dY + (size_t)row * rows.co, ((u >> 1) * 2 + (lane & 1)) * EPP, rows.co);
      }
    }
  };
  auto store_step = [&]() {
#pragma unroll
    for (int i = 0; i < XT; ++i) {
      const int u = wave + i * 4;
      if (XU >= 4 || u < XU) {
        const int pr = (u & 1) * 32 + (lane >> 1), c0 = ((u >> 1) * 2 + (lane & 1)) * EPP;
#pragma unroll
        for (int e = 0; e < EPP; ++e) {
          if constexpr (sizeof(S) == 2)
            *reinterpret_cast<u16 *>(&s_x[(c0 + e) * STRIDE + pr * 2]) =
                (u16)(xr[i][e >> 1] >> ((e & 1) * 16));
          else
            *reinterpret_cast<uint32_t *>(&s_x[(c0 + e) * STRIDE + pr * 4]) = xr[i][e];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < YT; ++i) {
      const int u = wave + i * 4;
      if (YU >= 4 || u < YU) {
        const int pr = (u & 1) * 32 + (lane >> 1), c0 = ((u >> 1) * 2 + (lane & 1)) * EPP;
#pragma unroll
        for (int e = 0; e < EPP; ++e) {
          if constexpr (sizeof(S) == 2)
            *reinterpret_cast<u16 *>(&s_y[(c0 + e) * STRIDE + pr * 2]) =
                (u16)(yr[i][e >> 1] >> ((e & 1) * 16));
          else
            *reinterpret_cast<uint32_t *>(&s_y[(c0 + e) * STRIDE + pr * 4]) = yr[i][e];
        }
      }
    }
  };

  for (int c_begin = 0; c_begin < run.length; c_begin += kFilterIndexChunk) {
    const int c_len = run.length - c_begin < kFilterIndexChunk ? run.length - c_begin : kFilterIndexChunk;
    __syncthreads();  // the previous chunk's indices are no longer read
    for (int t = tid; t < c_len; t += 256) {
      int i = -1, o = -1;
      const int p = run.at(c_begin + t);
      if (p < run.end) {
        i = in_col[p];
        o = out_col[p];
        if ((unsigned)i >= (unsigned)n_in || (unsigned)o >= (unsigned)n_out) i = o = -1;
      }
      s_in[t] = i;
      s_out[t] = o;
    }
    __syncthreads();
    fetch_step(0);
    for (int local = 0; local < c_len; local += SP) {
      __syncthreads();  // every wave has read the previous step's operands
      store_step();
      __syncthreads();
      if (local + SP < c_len) fetch_step(local + SP);
#pragma unroll
      for (int kb = 0; kb < SP / E::kChunk; ++kb) {
        vec8 bfr[COB];
#pragma unroll
        for (int b = 0; b < COB; ++b)
          bfr[b] = *reinterpret_cast<const vec8 *>(
              &s_y[(b * 16 + (lane & 15)) * STRIDE + kb * 64 + (lane >> 4) * 16]);
#pragma unroll
        for (int a = 0; a < CBW; ++a) {
          const int cb = wave + a * 4;
          if (cb < CI / 16) {
            const vec8 afr = *reinterpret_cast<const vec8 *>(
                &s_x[(cb * 16 + (lane & 15)) * STRIDE + kb * 64 + (lane >> 4) * 16]);
#pragma unroll
            for (int b = 0; b < COB; ++b) acc[a][b] = E::mfma(afr, bfr[b], acc[a][b]);
          }
        }
      }
    }
  }
  // lane holds rows 4*(lane/16)+v, column lane%16 of every 16 x 16 block
  float *tile = partial + (size_t)run.tile * CI * CO;
#pragma unroll
  for (int a = 0; a < CBW; ++a) {
    const int cb = wave + a * 4;
    if (cb < CI / 16) {
#pragma unroll
      for (int b = 0; b < COB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          tile[(size_t)(cb * 16 + 4 * (lane >> 4) + v) * CO + b * 16 + (lane & 15)] = acc[a][b][v];
    }
  }
}

// The same product for 17 to 128 channels on both sides and rows of whole 16-byte pieces (an LDS request takes one).  The
// gathered rows go from global memory straight into LDS as they are ([pair][channel], 16 bytes per lane), one step of SP
// pairs ahead into the other of two buffers.  No registers for staging, one barrier per step.  (Not bound by memory's
// latency: three, four or five buffers with as many steps under way gave the same times or, where fewer workgroups fit a CU,
// longer ones.  fp16, 128 x 128 channels, 2.85 M pairs of a 248 636-row scene, 108 us by counters: 0.69 GB come from behind the
// L2, 6.4 TB/s, where the two tensors have 0.13 GB; loaded data on its way into a CU 63 % busy, the matrix cores 35 %.)
//
// A row is asked for by the place where it begins, worked out once when the pair's index is staged: a buffer load answers
// a pair that is not there with zeros, and a load costs one addition in front of it (with a 64-bit address and a choice
// of a row of zeros, ten operations each, 128 x 128 channels of a 248 636-row scene took 161 us with the sums and not 147).
//
// 2-byte elements are transposed by the LDS read itself: `ds_read_b64_tr_b16` hands a lane four consecutive pairs of one
// channel; within 16 lanes, lane i supplies the address of 4 channels of pair i / 4 and lane j receives channel j of the
// four pairs.  Two such reads are one operand fragment.  A row's 16-byte pieces are stored permuted (piece ^ f(pair)),
// since rows lie a multiple of the bank width apart: f spreads the eight pairs that half a wavefront reads at once over
// all 64 banks.
constexpr int filterRowSwizzle(int row_bytes, int pair) {
  return row_bytes == 256 ? (((pair & 1) << 1) | ((pair & 2) << 1) | (pair & 8))
       : row_bytes == 128 ? ((pair & 2) | ((pair & 8) >> 1))
       : row_bytes == 64  ? ((pair & 8) >> 2)
                          : 0;
}

// An fp32 operand is one element a lane and needs no transposition: four-byte reads.  The pairs of a multiply are those of
// backwardFilterMfma (4 kq + s of 16 pairs), whose bits it gives.  The four rows a multiply reads at once have to meet
// all banks: a row's 64-byte chunks are permuted by bits 2 and 3 of its pair, and of rows of 128 bytes every second
// four stand in each other's places.
// Bound by the multiplies from 96 channels on (128 x 128: 223 us of them at the 144 TFLOP/s this instruction reaches) and by
// a step's round trip below.  us with the sums, 100 000-row scene, 0.98 M pairs, backwardFilterMfma / this:
//   32 x 32  53/41   48 x 48  137/66   64 x 64  141/92   68 x 36  247/106   64 x 96  260/133   96 x 96  377/211
//   32 x 128  190/106   128 x 128  362/300          and 3 000 rows, 20 000 pairs: 32 x 32  22/18   96 x 96  108/71
constexpr int floatRowChunk(int row_bytes, int pair) { return row_bytes >= 256 ? pair >> 2 & 3 : pair >> 3 & 1; }
constexpr int floatRowSlot(int row_bytes, int pair) { return row_bytes >= 256 ? pair : pair ^ (pair >> 2 & 1); }
// Where the row of pair 4 kq + q lies behind that of pair 4 kq.
__device__ __forceinline__ int floatStepPlace(int row_bytes, int q, int kq) {
  return row_bytes >= 256 ? q * row_bytes : (floatRowSlot(row_bytes, 4 * kq + q) - floatRowSlot(row_bytes, 4 * kq)) * row_bytes;
}

// Waves are laid out 2 x 2 over the blocks of dW[k], each with every second block of a side, so that the two waves of a
// side share the blocks that a row has.
// The place of a row that is not there: behind the end of every tensor (transposingReads) and, with a row's
// pieces added, below 2^32, so that the tensors may be twice as long as the gathered ones of the kernels above (2-byte output
// gradients of more than 2 GiB, which the kernel that stages rows through registers would take: 128 x 128 channels,
// 3.0 M pairs, 331 us, this one 224).
constexpr uint32_t kNoPlace = 0xfffffe00u;

template <typename E, int CI, int CO, int SP, bool WHOLE>
__global__ __launch_bounds__(256) void backwardFilterRows(
    const typename E::storage *X, const typename E::storage *dY, FilterGradRows lengths, const int32_t *pairs, int L,
    int x_col, int n_in, int n_out, int K, SliceTable tab, SliceOrder order, int total_slices,
    int slice_len, int shares, float *partial) {
  typedef typename E::vec8 vec8;
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef short v8i16 __attribute__((ext_vector_type(8)));
  constexpr int kSize = (int)sizeof(typename E::storage);
  constexpr bool kFloat = kSize == 4;
  static_assert(CI % 32 == 0 && CO % 32 == 0 && CI <= 128 && CO <= 128, "two row and column blocks per wave pair");
  static_assert(SP == 32 || SP == 64, "whole fragments, and whole steps in what a workgroup is given");
  constexpr int kIndexChunk = kFilterWalkChunk;  // a pair a thread
  constexpr int kChunkSteps = kIndexChunk / SP;
  static_assert(kIndexChunk == 256 && kChunkSteps > 2, "indices land in time (see the loop)");
  const FilterGradRows rows = WHOLE ? FilterGradRows{CI, CO} : lengths;
  constexpr int RBX = CI * kSize, RBY = CO * kSize;  // bytes per row
  constexpr int XN = SP * RBX / 1024;                // 1 KiB wave-loads per step, x first
  constexpr int LOADS = XN + SP * RBY / 1024;
  constexpr int MOST = (LOADS + 3) / 4;              // a wave's
  constexpr int AB = CI / 32, BB = CO / 32;          // 16-row / 16-column blocks per wave

  __shared__ __attribute__((aligned(1024))) char s_x[2][SP * RBX];
  __shared__ __attribute__((aligned(1024))) char s_y[2][SP * RBY];
  // where the x rows and the y rows of a chunk of pairs begin, and of the chunk after; kNoPlace: a pair that is not there
  __shared__ __attribute__((aligned(1024))) uint32_t s_at[2][2][kIndexChunk];

  const FilterRun run = runOfWorkgroup(tab, order, total_slices, slice_len, shares);
  if (run.k < 0) return;
  const int k = run.k;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wa = wave >> 1, wb = wave & 1;
  auto lds_of = [](const void *at) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)at; };
  auto words_of = [](const void *base, uint32_t bytes) {
    return u32x4{(uint32_t)reinterpret_cast<uintptr_t>(base), (uint32_t)(reinterpret_cast<uintptr_t>(base) >> 32), bytes,
                 0x00020000u};
  };
  const uint32_t x_lds = lds_of(&s_x[0][0]), y_lds = lds_of(&s_y[0][0]);
  const uint32_t index_lds = lds_of(&s_at[0][0][0]) + (uint32_t)wave * 256u;
  const uint32_t x_length = (uint32_t)(rows.ci * kSize), y_length = (uint32_t)(rows.co * kSize);  // zeros behind them
  const u32x4 x_words = words_of(X, (uint32_t)n_in * x_length), y_words = words_of(dY, (uint32_t)n_out * y_length);
  const u32x4 in_words = words_of(pairs + ((size_t)k * 2 + x_col) * L, (uint32_t)L * 4u);
  const u32x4 out_words = words_of(pairs + ((size_t)k * 2 + 1 - x_col) * L, (uint32_t)L * 4u);

  // blocks of 16 channels that the rows have, of this wave's
  const int blocks_a = WHOLE ? AB : ((rows.ci + 15) / 16 - wa + 1) / 2;
  const int blocks_b = WHOLE ? BB : ((rows.co + 15) / 16 - wb + 1) / 2;
  float4v acc[AB][BB];
#pragma unroll
  for (int a = 0; a < AB; ++a)
#pragma unroll
    for (int b = 0; b < BB; ++b) acc[a][b] = float4v{0.f, 0.f, 0.f, 0.f};

  // One step's rows into a buffer: a wave-load covers 1 KiB of it, lane l its bytes [16 l, 16 l + 16), i.e. a fixed (pair,
  // place) of the step.  Wave w issues loads w, w + 4, ...; all places are read first (one LDS latency a step,
  // not one a load).
  uint32_t piece[MOST];  // the piece of its row that a lane asks for, by load
  int pair_of[MOST];     // and the pair, in s_at[chunk & 1]
  bool of_x[MOST];
#pragma unroll
  for (int u = 0; u < MOST; ++u) {
    of_x[u] = u * 4 + 3 < XN || (u * 4 < XN && wave + u * 4 < XN);
    const int row_bytes = of_x[u] ? RBX : RBY;
    const int byte = ((of_x[u] ? 0 : -XN) + wave + u * 4) * 1024 + lane * 16;
    const int slot = byte / row_bytes % SP;
    const int pair = kFloat ? floatRowSlot(row_bytes, slot) : slot;
    const int moved = kFloat ? floatRowChunk(row_bytes, pair) * 4 : filterRowSwizzle(row_bytes, pair);
    piece[u] = (uint32_t)((byte % row_bytes / 16) ^ moved) * 16u;
    if (piece[u] >= (of_x[u] ? x_length : y_length)) piece[u] = kNoPlace;
    pair_of[u] = (of_x[u] ? 0 : kIndexChunk) + pair;
  }
  auto request_step = [&](int step, int buffer) {
    const uint32_t *at_step = &s_at[(step / kChunkSteps) & 1][0][(step % kChunkSteps) * SP];
    uint32_t at[MOST];
#pragma unroll
    for (int u = 0; u < MOST; ++u) at[u] = at_step[pair_of[u]];
#pragma unroll
    for (int u = 0; u < MOST; ++u) {
      // (a piece behind the row's end is nowhere, wherever the row begins)
      at[u] = WHOLE ? at[u] + piece[u] : __builtin_elementwise_min(__builtin_elementwise_add_sat(at[u], piece[u]), kNoPlace);
      asm volatile("" : "+v"(at[u]));
    }
#pragma unroll
    for (int u = 0; u < MOST; ++u) {
      if (LOADS % 4 != 0 && wave + u * 4 >= LOADS) break;
      if (of_x[u])
        requestRowsToLds(x_words, at[u], x_lds + (uint32_t)(buffer * (SP * RBX) + (wave + u * 4) * 1024));
      else
        requestRowsToLds(y_words, at[u], y_lds + (uint32_t)(buffer * (SP * RBY) + (wave + u * 4 - XN) * 1024));
    }
  };

  // Operand fragments: of 32 pairs of 2-byte elements, where lane (c, kq) receives the pairs 8 kq + (0..7) of channel
  // 16 block + c, or, element by element, of 16 pairs in fp32, where multiply s takes its pair 4 kq + s.  (What is
  // permuted by pair is the same for the four pairs and for the next fragment.)
  const int sub = lane & 15, kq = lane >> 4;
  auto fragment_place = [&](int row_bytes, int block) -> int {
    if (kFloat)
      return floatRowSlot(row_bytes, 4 * kq) * row_bytes + (block ^ floatRowChunk(row_bytes, 4 * kq)) * 64 + sub * 4;
    const int pair = 8 * kq + (sub >> 2);
    const int place = (block * 2 + ((sub & 3) >> 1)) ^ filterRowSwizzle(row_bytes, pair);
    return pair * row_bytes + place * 16 + (sub & 1) * 8;
  };
  const char *x_frag[AB], *y_frag[BB];  // in the first buffer
#pragma unroll
  for (int a = 0; a < AB; ++a) x_frag[a] = &s_x[0][0] + fragment_place(RBX, wa + 2 * a);
#pragma unroll
  for (int b = 0; b < BB; ++b) y_frag[b] = &s_y[0][0] + fragment_place(RBY, wb + 2 * b);
  auto fragment = [&](const char *at, int row_bytes) -> vec8 {
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) v4i16 *)(at));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) v4i16 *)(at + 4 * row_bytes));
    const v8i16 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(vec8, both);
  };
  auto multiply = [&](int buffer) {
    const int x_at = buffer * (SP * RBX), y_at = buffer * (SP * RBY);
    if constexpr (kFloat) {
#pragma unroll
      for (int kb = 0; kb < SP / 16; ++kb) {
        float xs[4][AB], ys[4][BB];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int a = 0; a < AB; ++a)
            xs[q][a] = *reinterpret_cast<const float *>(x_frag[a] + x_at + kb * 16 * RBX + floatStepPlace(RBX, q, kq));
#pragma unroll
          for (int b = 0; b < BB; ++b)
            ys[q][b] = *reinterpret_cast<const float *>(y_frag[b] + y_at + kb * 16 * RBY + floatStepPlace(RBY, q, kq));
        }
        // (the blocks that a row does not have are zeros in LDS; their multiplies are left out, behind the reads: a branch
        // between reads and multiplies made small layers slower)
#pragma unroll
        for (int a = 0; a < AB; ++a) {
          if (a >= blocks_a) break;
#pragma unroll
          for (int b = 0; b < BB; ++b) {
            if (b >= blocks_b) break;
#pragma unroll
            for (int q = 0; q < 4; ++q)
              acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[q][a], ys[q][b], acc[a][b], 0, 0, 0);
          }
        }
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < SP / 32; ++kb) {
        vec8 bfr[BB];
#pragma unroll
        for (int b = 0; b < BB; ++b) bfr[b] = fragment(y_frag[b] + y_at + kb * 32 * RBY, RBY);
#pragma unroll
        for (int a = 0; a < AB; ++a) {
          const vec8 afr = fragment(x_frag[a] + x_at + kb * 32 * RBX, RBX);
#pragma unroll
          for (int b = 0; b < BB; ++b) acc[a][b] = E::mfma(afr, bfr[b], acc[a][b]);
        }
      }
    }
  };

  // A chunk's indices: a thread's own, to LDS as they are; then checked, and places where they stood.
  auto request_indices = [&](int chunk) {
    const uint32_t at = (uint32_t)run.at(chunk * kIndexChunk + tid) * 4u;  // (behind the list: zeros, checked below)
    const uint32_t to = index_lds + (uint32_t)(chunk & 1) * (2 * kIndexChunk * 4);
    requestWordsToLds(in_words, at, to);
    requestWordsToLds(out_words, at, to + kIndexChunk * 4);
  };
  auto place_indices = [&](int chunk) {
    uint32_t &in = s_at[chunk & 1][0][tid], &out = s_at[chunk & 1][1][tid];
    const uint32_t i = in, o = out;
    const bool there = run.at(chunk * kIndexChunk + tid) < run.end && i < (uint32_t)n_in && o < (uint32_t)n_out;
    in = there ? i * x_length : kNoPlace;
    out = there ? o * y_length : kNoPlace;
  };

  const int steps = run.length / SP;
  if (steps > 0) {
    request_indices(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    place_indices(0);
    ldsBarrier();
    request_step(0, 0);
  }
  for (int step = 0; step < steps; ++step) {
    const int cur = step & 1;
    // this step's rows have landed, and every wave has left the buffers of the step before
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ldsBarrier();
    // The chunk after this one: its indices are requested at the chunk's first step (the places they come over were last
    // read two steps before) and are places one barrier before the chunk's last step asks for the next one's first rows.
    const int in_chunk = step % kChunkSteps, chunk = step / kChunkSteps;
    const bool chunk_follows = (chunk + 1) * kChunkSteps < steps;
    if (in_chunk == 0 && chunk_follows) request_indices(chunk + 1);
    // (all requests first: they have one step's multiplies to land; the other workgroups' requests wait for these
    // multiplies)
    if (step + 1 < steps) request_step(step + 1, cur ^ 1);
    __builtin_amdgcn_s_setprio(1);
    multiply(cur);
    __builtin_amdgcn_s_setprio(0);
    if (in_chunk == kChunkSteps - 2 && chunk_follows) place_indices(chunk + 1);
  }
  // lane holds rows 4*(lane/16)+v, column lane%16 of every 16 x 16 block
  float *const sums = partial + (size_t)run.tile * CI * CO;
#pragma unroll
  for (int a = 0; a < AB; ++a)
#pragma unroll
    for (int b = 0; b < BB; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        sums[(size_t)((wa + 2 * a) * 16 + 4 * (lane >> 4) + v) * CO + (wb + 2 * b) * 16 + (lane & 15)] =
            acc[a][b][v];
}

// dW[k] = sum of the offset's partial tiles, rounded once.  A block adds 256
// consecutive elements (four per lane): wave g of 16 takes the slices g, g+16, ...
// in eight independent running sums, the sums are combined pairwise in a fixed
// order, so the result depends on the slice count only, never on timing.
constexpr int kSliceSumWaves = 16;
template <typename E>
__global__ __launch_bounds__(64 * kSliceSumWaves) void sliceSum(const float *partial,
                                                                SliceTable tab, int slice_len,
                                                                int tile_elems, int tile_co, FilterGradRows rows,
                                                                GradLayout lay,
                                                                typename E::storage *dW) {
  constexpr int W = kSliceSumWaves;
  __shared__ float4v s_part[W][64];
  const int k = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int g = threadIdx.x >> 6;
  const int e = (blockIdx.x * 64 + lane) * 4;  // tile_elems is a multiple of 256
  const int slices = tab.tiles[k];
  float4v acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = float4v{0.f, 0.f, 0.f, 0.f};
  if (e < tile_elems) {
    const float *src = partial + (size_t)tab.first[k] * tile_elems + e;
    for (int i0 = g; i0 < slices; i0 += 8 * W) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = i0 + W * u;
        if (i < slices) acc[u] += *reinterpret_cast<const float4v *>(src + (size_t)i * tile_elems);
      }
    }
  }
  s_part[g][lane] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  __syncthreads();
  if (g == 0 && e < tile_elems) {
    float4v t[W];
#pragma unroll
    for (int i = 0; i < W; ++i) t[i] = s_part[i][lane];
#pragma unroll
    for (int span = 1; span < W; span *= 2)
#pragma unroll
      for (int i = 0; i < W; i += 2 * span) t[i] += t[i + span];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ci = (e + v) / tile_co, co = (e + v) % tile_co;
      if (ci < rows.ci && co < rows.co) E::store(dW + gradOffset(lay, k, ci, co), t[0][v]);
    }
  }
}

// The same sum on a flat grid for filters with many offsets, where most offsets own
// a handful of slices and a 1024-thread workgroup per 256 elements is mostly idle
// waves (at 125 offsets x 128 x 128: 8000 workgroups, dispatch-bound).  An offset with
// at most 16 slices is "thin": each wave sums one 256-element chunk on its own, so a
// workgroup covers 16 chunks and needs no barrier.  The additions are those of
// sliceSum in the same order (a wave's partial there is 0 + slice g when the offset
// has at most 16 slices), so both kernels give the same bits.
struct SumGrid {
  int first[kMaxInlineK];  // workgroups in front of the offset's first one
};
constexpr int kThinSlices = kSliceSumWaves;

template <typename E>
__global__ __launch_bounds__(64 * kSliceSumWaves) void sliceSumFlat(const float *partial,
                                                                    SliceTable tab, SumGrid grid,
                                                                    int K, int slice_len,
                                                                    int tile_elems, int tile_co, FilterGradRows rows,
                                                                    GradLayout lay,
                                                                    typename E::storage *dW) {
  constexpr int W = kSliceSumWaves;
  __shared__ float4v s_part[W][64];
  // last offset whose first workgroup is not behind this one
  int lo = 0, hi = K - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (grid.first[mid] <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
  }
  const int k = lo;
  const int chunk = blockIdx.x - grid.first[k];
  const int lane = threadIdx.x & 63;
  const int g = threadIdx.x >> 6;
  const int slices = tab.tiles[k];
  const float *tiles = partial + (size_t)tab.first[k] * tile_elems;
  if (slices <= kThinSlices) {
    const int e = ((chunk * W + g) * 64 + lane) * 4;
    if (e >= tile_elems) return;
    float4v t[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      t[i] = float4v{0.f, 0.f, 0.f, 0.f};
      if (i < slices) t[i] += *reinterpret_cast<const float4v *>(tiles + (size_t)i * tile_elems + e);
    }
#pragma unroll
    for (int span = 1; span < W; span *= 2)
#pragma unroll
      for (int i = 0; i < W; i += 2 * span) t[i] += t[i + span];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ci = (e + v) / tile_co, co = (e + v) % tile_co;
      if (ci < rows.ci && co < rows.co) E::store(dW + gradOffset(lay, k, ci, co), t[0][v]);
    }
    return;
  }
  const int e = (chunk * 64 + lane) * 4;
  float4v acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = float4v{0.f, 0.f, 0.f, 0.f};
  {
    const float *src = tiles + e;
    for (int i0 = g; i0 < slices; i0 += 8 * W) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = i0 + W * u;
        if (i < slices) acc[u] += *reinterpret_cast<const float4v *>(src + (size_t)i * tile_elems);
      }
    }
  }
  s_part[g][lane] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  __syncthreads();
  if (g == 0) {
    float4v t[W];
#pragma unroll
    for (int i = 0; i < W; ++i) t[i] = s_part[i][lane];
#pragma unroll
    for (int span = 1; span < W; span *= 2)
#pragma unroll
      for (int i = 0; i < W; i += 2 * span) t[i] += t[i + span];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ci = (e + v) / tile_co, co = (e + v) % tile_co;
      if (ci < rows.ci && co < rows.co) E::store(dW + gradOffset(lay, k, ci, co), t[0][v]);
    }
  }
}

// ---- host side -----------------------------------------------------------------------

inline size_t alignUp(size_t v, size_t a = 256) { return (v + a - 1) / a * a; }

// Workspace blocks are carved from the caller's pointer rounded up to 256 bytes;
// the reported sizes include that slack.
constexpr size_t kBaseAlign = 256;
inline char *alignPtr(void *p) {
  if (p == nullptr) return nullptr;
  return reinterpret_cast<char *>(alignUp(reinterpret_cast<uintptr_t>(p), kBaseAlign));
}

inline int gridFor(size_t n, int cap = 8192) {
  size_t b = (n + 255) / 256;
  return (int)(b < 1 ? 1 : (b > (size_t)cap ? (size_t)cap : b));
}

// The backward filter's partial tiles are summed on the flat grid from this many
// workgroups on (or as the handle's kernel choice says; the two kernels give the same bits).
constexpr int kFlatSumFromBlocks = 2048;

// The matrix-core kernels are compiled for 16, 32, 64 and 128 channels (fp16/bf16: 16x16x32
// MFMA, 16 channels as half-filled fragments; float: 16x16x4); a tensor of up to 128 channels
// runs on the next of these.
int paddedChannels(int c) { return c <= 16 ? 16 : (c <= 32 ? 32 : (c <= 64 ? 64 : 128)); }
bool mfmaShapeOk(int Q, int C) { return Q >= 1 && Q <= 128 && C >= 1 && C <= 128; }

// They read rows in 16-byte pieces.  Rows of another length (4 or 5 point features, 12 channels
// of a 2-byte type) are copied to padded rows in the workspace first, by workgroups of the
// launch that prepares the filter.
int paddedRowBytes(ElemType t, int channels) { return (channels * (int)elemSize(t) + 15) / 16 * 16; }
bool rowsNeedPadding(ElemType t, int channels) { return channels * (int)elemSize(t) % 16 != 0; }

struct GatherDims {
  int R;       // result rows
  int n_src;   // rows of the gathered tensor
  int Q;       // reduction channels
  int C;       // result channels
  int q_padded, c_padded;  // of the matrix-core instance
  int row_col, src_col;
  bool filter_forward;  // B(k, q, c) = W(k, ci = q, co = c); otherwise its transpose
};

GatherDims gatherDims(const ConvProblem &p, GatherDirection dir) {
  GatherDims d;
  d.filter_forward = dir == GatherDirection::kForward;
  if (d.filter_forward) {
    d.Q = p.Ci; d.C = p.Co;
  } else {
    d.Q = p.Co; d.C = p.Ci;
  }
  d.q_padded = paddedChannels(d.Q);
  d.c_padded = paddedChannels(d.C);
  // The result rows are the pair column the operator writes through: column 1
  // for forward, column 0 for backward data, and the other way round for an
  // inverse convolution, which runs its partner's rulebook backwards.
  if (d.filter_forward != p.inverse) {
    d.R = p.num_out; d.n_src = p.L; d.row_col = 1; d.src_col = 0;
  } else {
    d.R = p.L; d.n_src = p.num_out; d.row_col = 0; d.src_col = 1;
  }
  return d;
}

// The list kernels take the per-offset tables by value and are asked for only when the
// caller has reason to believe the result-row column in order; a row map announced for
// the call is used instead.
bool listsUsable(const ConvProblem &p, const GatherDims &d) {
  (void)d;
  return p.list_trust != ListTrust::kNone && p.K <= kMaxInlineK && p.row_map == nullptr;
}

struct GatherWorkspace {
  int32_t *cuts = nullptr;              // [K, tiles + 1] cut positions of the pair lists
  unsigned long long *verdict = nullptr;
  int32_t *dev_counts = nullptr;
  int32_t *filled = nullptr;  // map slots the gather kernel's workgroups found filled
  int32_t *accepted = nullptr;  // pairs the map scatter's workgroups put into the map
  int map_rows = 0;           // result rows one map holds: the rows of a chunk
  int32_t *shadow = nullptr;  // repairLostPairs' scratch, touched only when pairs collide
  int32_t *pool_row = nullptr;
  float *pool = nullptr;
  int32_t *map = nullptr;
  void *packed = nullptr;
  void *padded_rows = nullptr;  // the gathered tensor with rows of whole 16-byte pieces
  size_t bytes = 0;
};

// Workgroups of repairLostPairs: one per window of result rows, kRepairBlocks at most.
int repairBlocks(int R) {
  const int windows = (R + kRepairPoolRows - 1) / kRepairPoolRows;
  return windows < 1 ? 1 : (windows > kRepairBlocks ? kRepairBlocks : windows);
}

// Entries of the `accepted` array the scatter kernels may write for K offsets of up to L pairs.
size_t scatterBlocksBound(int K, int L) {
  const size_t flat = (size_t)K * ((size_t)L / 256 + 1);
  const size_t grid = (size_t)K * 1024;
  return flat > grid ? flat : grid;
}

// The row map is built and used for a chunk of result rows at a time, so that it stays
// below kMapChunkBytes however many offsets and rows there are (a multiple of the repair
// window, hence of every tile height).
constexpr size_t kMapChunkBytes = 64u << 20;
int mapChunkRows(int K, int R) {
  size_t rows = kMapChunkBytes / ((size_t)K * 4);
  rows = rows / kRepairPoolRows * kRepairPoolRows;
  if (rows < (size_t)kRepairPoolRows) rows = kRepairPoolRows;
  return rows < (size_t)R ? (int)rows : R;
}

GatherWorkspace carveGather(const ConvProblem &p, const GatherDims &d, void *base) {
  GatherWorkspace ws;
  ws.map_rows = mapChunkRows(p.K, d.R);
  char *ptr = alignPtr(base);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *r = ptr ? ptr + off : nullptr;
    off += alignUp(bytes);
    return r;
  };
  if (p.K > kMaxInlineK) ws.dev_counts = reinterpret_cast<int32_t *>(take((size_t)p.K * 4));
  if (p.K <= kMaxInlineK) {
    // tiles of the narrowest kind (64 rows) bound the table
    ws.cuts = reinterpret_cast<int32_t *>(take((size_t)p.K * ((size_t)d.R / 64 + 2) * 4));
    ws.verdict = reinterpret_cast<unsigned long long *>(take(8));
  }
  ws.filled = reinterpret_cast<int32_t *>(take(((size_t)d.R / 32 + 16) * 4));
  ws.accepted = reinterpret_cast<int32_t *>(take(scatterBlocksBound(p.K, p.L) * 4));
  ws.shadow = reinterpret_cast<int32_t *>(take((size_t)ws.map_rows * 4));
  const size_t repair_blocks = (size_t)repairBlocks(ws.map_rows);
  ws.pool_row = reinterpret_cast<int32_t *>(take(repair_blocks * kRepairPoolRows * 4));
  ws.pool = reinterpret_cast<float *>(take(repair_blocks * kRepairPoolRows * d.C * 4));
  ws.map = reinterpret_cast<int32_t *>(take((size_t)p.K * ws.map_rows * 4));
  if (mfmaShapeOk(d.Q, d.C)) {
    // reduction channels are padded to whole 16-byte fragments (32 for the 2-byte types)
    const size_t chunk = 64 / elemSize(p.dtype);
    const size_t q_padded = ((size_t)d.q_padded + chunk - 1) / chunk * chunk;
    ws.packed = take((size_t)p.K * q_padded * d.c_padded * elemSize(p.dtype) + ((size_t)p.K + 1) * 8);
    if (rowsNeedPadding(p.dtype, d.Q)) ws.padded_rows = take((size_t)d.n_src * paddedRowBytes(p.dtype, d.Q));
  }
  ws.bytes = off + kBaseAlign;
  return ws;
}

// Writes n counts, carried in the kernel arguments, to dst.
__global__ void storeCounts(OffsetCounts c, int n, int32_t *dst) {
  const int i = threadIdx.x;
  if (i < n) dst[i] = c.n[i];
}

// Fills the by-value counts (K <= kMaxInlineK) or puts them into device memory: kMaxInlineK
// counts ride in the arguments of one small launch each, so the host neither allocates nor
// waits, and the call can be captured into a graph like any other.
hipError_t prepareCounts(const LaunchCtx &lc, const ConvProblem &p, OffsetCounts *inl,
                         int32_t *dev_counts, int *max_count) {
  auto clamped = [&](int k) {
    const int64_t n = p.indice_num[k];
    return (int)(n < 0 ? 0 : (n > p.L ? p.L : n));
  };
  int mx = 0;
  for (int k = 0; k < p.K; ++k) mx = clamped(k) > mx ? clamped(k) : mx;
  *max_count = mx;
  for (int k = 0; k < kMaxInlineK; ++k) inl->n[k] = 0;
  if (p.K <= kMaxInlineK) {
    for (int k = 0; k < p.K; ++k) inl->n[k] = clamped(k);
    return hipSuccess;
  }
  for (int k0 = 0; k0 < p.K; k0 += kMaxInlineK) {
    OffsetCounts part;
    const int n = p.K - k0 < kMaxInlineK ? p.K - k0 : kMaxInlineK;
    for (int i = 0; i < kMaxInlineK; ++i) part.n[i] = i < n ? clamped(k0 + i) : 0;
    storeCounts<<<1, kMaxInlineK, 0, lc.stream>>>(part, n, dev_counts + k0);
  }
  return hipGetLastError();
}

// A 128-column result with few pairs per (64-row tile, offset) runs as two
// 64-column halves over 128-row tiles: twice the entries in every block for
// the same accumulator size, at the price of gathering each row twice.
int mfmaTileCols(const ConvProblem &p, const GatherDims &d) {
  if (d.c_padded != 128) return d.c_padded;
  double pairs = 0;
  for (int k = 0; k < p.K; ++k) pairs += (double)p.indice_num[k];
  const double per_tile_offset = pairs * mfmaTileRows(128) / ((double)d.R * p.K);
  return per_tile_offset < 8.0 ? 64 : 128;
}

// Workgroups along x: tiles rounded up to a multiple of the XCD count.
int mfmaGridX(int R, int tile_cols) {
  const int tr = mfmaTileRows(tile_cols);
  return ((R + tr - 1) / tr + 7) / 8 * 8;
}
int denseGridX(int R) { return ((R + kDenseRows - 1) / kDenseRows + 7) / 8 * 8; }

template <typename E, int Q, int C, typename SRC>
void launchMfmaInstance(const LaunchCtx &lc, const void *A, const ConvRows &rows, const void *packed,
                        const SRC &source, int R, int K, void *result) {
  constexpr int NT = mfmaThreads(C);
  const dim3 grid(mfmaGridX(R, C), (rows.c + C - 1) / C);
  lc.begin("gatherConvMfma");
  gatherConvMfma<E, Q, C, SRC><<<grid, NT, 0, lc.stream>>>(
      static_cast<const typename E::storage *>(A), rows,
      static_cast<const typename E::storage *>(packed), source, R, K,
      static_cast<typename E::storage *>(result));
  lc.end();
}

// `tile_cols` result columns per workgroup: a narrower tile has more rows, so sparse
// rulebooks fill their 16-pair blocks better.
template <typename E, int Q, typename SRC>
void launchMfmaByC(const LaunchCtx &lc, int tile_cols, const void *A, const ConvRows &rows, const void *packed,
                   const SRC &source, int R, int K, void *result) {
  switch (tile_cols) {
    case 16: launchMfmaInstance<E, Q, 16, SRC>(lc, A, rows, packed, source, R, K, result); break;
    case 32: launchMfmaInstance<E, Q, 32, SRC>(lc, A, rows, packed, source, R, K, result); break;
    case 64: launchMfmaInstance<E, Q, 64, SRC>(lc, A, rows, packed, source, R, K, result); break;
    case 128: launchMfmaInstance<E, Q, 128, SRC>(lc, A, rows, packed, source, R, K, result); break;
    default: break;
  }
}

template <typename E, typename SRC>
void launchMfma(const LaunchCtx &lc, int q_padded, int tile_cols, const void *A, const ConvRows &rows,
                const void *packed, const SRC &source, int R, int K, void *result) {
  switch (q_padded) {
    case 16: launchMfmaByC<E, 16, SRC>(lc, tile_cols, A, rows, packed, source, R, K, result); break;
    case 32: launchMfmaByC<E, 32, SRC>(lc, tile_cols, A, rows, packed, source, R, K, result); break;
    case 64: launchMfmaByC<E, 64, SRC>(lc, tile_cols, A, rows, packed, source, R, K, result); break;
    case 128: launchMfmaByC<E, 128, SRC>(lc, tile_cols, A, rows, packed, source, R, K, result); break;
    default: break;
  }
}

template <typename E, int Q, int C>
void launchWaveInstance(const LaunchCtx &lc, const void *A, const ConvRows &rows, const void *packed,
                        const SegmentSource &source, int R, int K, void *result) {
  if constexpr (waveKernelShape((int)sizeof(typename E::storage), Q, C)) {
    const int grid = ((R + kWaveTileRows - 1) / kWaveTileRows + 7) / 8 * 8;
    lc.begin("gatherConvWave");
    const bool whole = rows.q == Q && rows.c == C;
    auto kernel = whole ? gatherConvWave<E, Q, C, true> : gatherConvWave<E, Q, C, false>;
    kernel<<<grid, 64, 0, lc.stream>>>(
        static_cast<const typename E::storage *>(A), rows, static_cast<const typename E::storage *>(packed),
        source, R, K, static_cast<typename E::storage *>(result));
    lc.end();
  }
}

template <typename E>
void launchWave(const LaunchCtx &lc, int q_padded, const void *A, const ConvRows &rows, const void *packed,
                const SegmentSource &source, int R, int K, void *result) {
#define WAVE_CASE(q)                                                                      \
  case q:                                                                                 \
    if (rows.c_padded == 16) launchWaveInstance<E, q, 16>(lc, A, rows, packed, source, R, K, result); \
    else launchWaveInstance<E, q, 32>(lc, A, rows, packed, source, R, K, result);         \
    break;
  switch (q_padded) {
    WAVE_CASE(16)
    WAVE_CASE(32)
    WAVE_CASE(64)
    WAVE_CASE(128)
    default: break;
  }
#undef WAVE_CASE
}

// Workgroups along x of the tall-tile kernel: tiles rounded up to a multiple of the XCD count.
int tallGridX(int R, int tile_rows) { return ((R + tile_rows - 1) / tile_rows + 7) / 8 * 8; }

template <typename E, int Q, typename SRC>
void launchTallInstance(const LaunchCtx &lc, const void *A, uint32_t a_size, const ConvRows &rows, const void *packed,
                        const SRC &source, int tile_rows, int R, int K, void *result) {
  constexpr int S = (int)sizeof(typename E::storage);
  constexpr int TR = tallRows(Q * S);
  auto launch = [&](auto kernel, int threads) {
    const dim3 grid(tallGridX(R, tile_rows), (rows.c + kTallCols - 1) / kTallCols);
    lc.begin(tile_rows == 512 && TR == 256 ? "gatherConvTall512" : "gatherConvTall");
    kernel<<<grid, threads, 0, lc.stream>>>(static_cast<const typename E::storage *>(A), a_size, rows,
                                            static_cast<const typename E::storage *>(packed), source, R, K,
                                            static_cast<typename E::storage *>(result));
    lc.end();
  };
  if constexpr (SRC::kSegments && TR == 256) {
    if (tile_rows == 128) return launch(gatherConvTall<E, Q, kTallCols, 128, SRC>, tallThreads(S, Q * S, 128));
    if constexpr (S == 2)
      if (tile_rows == 512) return launch(gatherConvTall<E, Q, kTallCols, 512, SRC>, tallThreads(S, Q * S, 512));
  }
  launch(gatherConvTall<E, Q, kTallCols, TR, SRC>, tallThreads(S, Q * S, TR));
}

// Channels of the instance for rows of q_padded channels (16 channels of a 2-byte type are half a fragment,
// packed like a whole one).
int tallQ(ElemType t, int q_padded) { return t != ElemType::kFloat && q_padded < 32 ? 32 : q_padded; }

template <typename E, typename SRC>
void launchTall(const LaunchCtx &lc, int q, const void *A, int n_src, const ConvRows &rows, const void *packed,
                const SRC &source, int tile_rows, int R, int K, void *result) {
  const uint32_t a_size = (uint32_t)n_src * (uint32_t)rows.row_bytes;
  switch (q) {
    case 16:
      if constexpr (std::is_same<E, FloatElem>::value)
        launchTallInstance<E, 16, SRC>(lc, A, a_size, rows, packed, source, tile_rows, R, K, result);
      break;
    case 32: launchTallInstance<E, 32, SRC>(lc, A, a_size, rows, packed, source, tile_rows, R, K, result); break;
    case 64: launchTallInstance<E, 64, SRC>(lc, A, a_size, rows, packed, source, tile_rows, R, K, result); break;
    case 128: launchTallInstance<E, 128, SRC>(lc, A, a_size, rows, packed, source, tile_rows, R, K, result); break;
    default: break;
  }
}

bool useWaveKernel(const LaunchCtx &lc, ElemType t, int Q, int C) {
  if (lc.choices.wave_per_tile == 0) return false;
  return waveKernelShape((int)elemSize(t), Q, C);
}

// The register-accumulating kernel addresses the gathered tensor with 32-bit byte offsets: tensors of
// 2 GiB and more take the pair-list kernels.
bool denseShapeOk(const ConvProblem &p, const GatherDims &d) {
  // (fp32 rows of more than 64 channels have no instance)
  if (p.dtype == ElemType::kFloat && d.Q > 64) return false;
  return (uint64_t)d.n_src * (uint64_t)paddedRowBytes(p.dtype, d.Q) < (uint64_t)kNoRow;
}

// Pair lists of so few rows that tiles of 128 do not outnumber the CUs run in those (tallHalfTiles): the
// launch is one tile long then, and half a tile is half as many blocks.  us of gatherConvMfma / tiles of 256 /
// of 128, fp16 64 -> 64, 128 -> 128 and fp32 64 -> 64:
//   3x3x3 in boxes      4 k rows 15/18/12.9, 19/22/15.5, 28/35/23.2;    16 k 15/19/13.5, 21/24/17.2, 30/37/24.2
//         strewn        16 k 13/14/11.9, 16/17/14.6, 23/24/20.5;        32 k 14/15/12.7, (22/19/21.0), 26/27/21.8
//   5x5x5 in boxes      4 k 41/39/29.4, 57/51/37.9, 88/88/64.3;         16 k 42/47/33.6, 59/58/41.6, 91/99/66.8
//   2x2x2 stride 2      12 k 11/13/10.4, 13/14/11.6, 17/20/15.4;        3x3x3 stride 2, 26 k 15/17/13.7, -, 28/31/23.2
// With two tiles on some CUs the tall ones win or lose with the fill (45 k strewn 17.1/15.8/17.1, in boxes
// 24/26/22.5), so gatherConvMfma stays there; over row maps tiles of 128 are no faster than it.
// More than 32 offsets run in them from the first row on: with tiles of 256, which take all longer lists of so
// many offsets, a layer of few rows is slower than one of more, and than gatherConvMfma at 63 offsets:
//   5x5x5 in boxes      64 rows 37/26/25.7, 52/33/32.8, 78/57/56;       1 k 43/41/28.5, 59/52/37.0, 89/90/63.7
//                       3 k 42/42/32.5, 57/53/37.7, 90/92/65.0
//         strewn        128 rows 22/13/12.8, 24/13/12.3, 27/16/15.9;    2 k 36/32/25.5, 46/36/31.0, 70/63/52.7
//   3x3x7 in boxes      64 rows 24/17/16.8, 32/21/20.3, 47/34/33.7;     3 k 26/29/20.7, 34/36/22.4, 53/62/37.0
// Up to 32 offsets gatherConvMfma stays below 4096 rows.  These tiles are ahead there too (3x3x3 in boxes, 64 rows
// 13/12/11.4, 16/13/13.1, 23/20/19.5; 1 k 14/18/12.8, 19/22/14.4, 27/35/21.5; 3 k 15/18/12.9, 19/21/15.1, 28/35/22.9),
// by 1 to 6 us of a layer's 50 to 100: a lower line is open, and no measurement speaks for this one.
constexpr int kTallFewRows = 128 * 256;  // times 64 result columns
constexpr int kTallFewestRows = 4096;    // with up to kTallFewOffsets offsets
constexpr int kTallFewOffsets = 32;
bool tallHalfTiles(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d) {
  return lc.choices.tall_tiles < 0 && (p.K > kTallFewOffsets || d.R >= kTallFewestRows) &&
         tallRows(d.q_padded * (int)elemSize(p.dtype)) == 256 && (int64_t)d.R * (d.c_padded / 64) <= kTallFewRows;
}

// Rows of a tall tile.  Many offsets of short lists (the filters of 125 at 128 x 128 channels are 4 MB, and every tile reads
// them): 512 rows with two teams of multiplying waves, for 2-byte types and rows of 65 channels up; one of 33 to 64 still
// gains, one of 32 does not.  us of tiles of 256 / 512 rows, fp16, surfaces, 5x5x5:
//   128 -> 128   400 k rows 449/360   200 k 246/212   50 k 73/54      128 -> 64   400 k 235/193   50 k 54/50
//    96 -> 96    400 k rows 410/349   100 k 138/117                    64 -> 64   400 k 165/150   100 k 71/65   50 k 43/42
//    32 -> 64    400 k rows 139/142   50 k 37/41
//   3x3x3, clustered: 128 -> 128  400 k 243/232   200 k 117/118;  64 -> 64  400 k 99/104   60 k 23/25;  uniform, 200 k:
//   128 -> 128  69/78;  2x2x2 stride 2, 177 k rows: 128 -> 128  55/60: up to 32 offsets stay with 256.
// A CU has one such tile at a time and nothing to do in its round trips, and a launch lasts as long as its heaviest tile:
// fewer workgroups than half the CUs, or many pairs a row, favour two tiles of 256.  us, 5x5x5, by pairs a row, with the
// filter's packing:
//   by workgroups  128 -> 64, gradient of stride 2 (15 pairs)  98 workgroups 105/132   196 200/164   390 373/324
//                  128 -> 64, stride 2 of a scene (5 to 8)     116 113/145   258 236/235   374 276/288   839 526/468
//                  128 -> 64, stride 2 of surfaces (1)         140 61/44     265 89/78     96 -> 96, scene (4)  140 108/136
//                  64 -> 128, surfaces (2) 80 42/39   196 53/44    stride 2 of a thinned scene (3) 106 43/48
//   64 channels    64 -> 64   surfaces (3) 391 workgroups 110/103   clustered (8) 391 152/152  (11) 782 311/296
//                             stride 2, strewn (2.6) 559 100/95   thinned scene (3.6) 422 109/117   scene (7) 839 355/368
//                             gradient of stride 2 (15) 391 193/213         64 -> 128  782 305/328
//                  64 -> 128  stride 2, strewn (2.6) 1118 163/150  thinned scene (4) 316 89/100   scene (6) 516 214/230
int tallTileRows(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d, int tall_q, bool lists) {
  const int row_bytes = tall_q * (int)elemSize(p.dtype);
  if (lists && tallHalfTiles(lc, p, d)) return 128;
  if (!lists || p.K <= kTallFewOffsets || elemSize(p.dtype) != 2 || row_bytes < 128) return tallRows(row_bytes);
  if (lc.choices.tall_tiles == 1) return 512;
  double pairs = 0, largest = 0;
  for (int k = 0; k < p.K; ++k) {
    pairs += (double)p.indice_num[k];
    largest = (double)p.indice_num[k] > largest ? (double)p.indice_num[k] : largest;
  }
  const int64_t workgroups = ((int64_t)d.R + 511) / 512 * (d.c_padded / kTallCols);
  const bool submanifold = largest >= 0.9 * d.R;  // (every row is in the centre's pairs)
  const int64_t enough = pairs < 2.2 * d.R ? 64 : pairs < 4.0 * d.R || row_bytes < 256 ? 128 : 160;
  const bool tall = workgroups >= enough && (row_bytes >= 256 || submanifold || pairs < 3.0 * d.R);
  return tall ? 512 : tallRows(row_bytes);
}

bool useTallKernel(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d, bool lists) {
  // (rows are addressed with 32-bit byte offsets; results of up to 32 columns have kernels of their own)
  if (d.c_padded < 64 || (uint64_t)d.n_src * (uint64_t)paddedRowBytes(p.dtype, d.Q) >= (uint64_t)kNoRow) return false;
  if (lc.choices.tall_tiles >= 0) return lc.choices.tall_tiles == 1;
  // What a tile of 256 rows saves is filters (one for the pairs of 256 rows instead of 128) and the second,
  // partly filled round of tiles; what it costs is that a CU's two tiles are long chains, so few rows
  // leave CUs idle, and that many pairs a tile do not fit its lists at once.  us of gatherConvMfma
  // against this kernel, 3x3x3 unless noted:
  //   fp16  64 -> 64, rows strewn              8 k 11/11,  60 k 13.6/13.4, 200 k 37/28;  5x5x5 60 k 31/20, 200 k 110/59
  //        128 -> 128, in boxes               12 k 17/18,  60 k 42/29,     200 k 149/104; 5x5x5 200 k 506/311
  //         64 -> 64, strided, 97 k rows of a scene, 0.196 filled: 61/64; 36 k, 0.204: 29/41
  //   fp32  64 -> 128, strided, strewn         60 k 180/92, 120 k 331/158; 64 -> 64, 12 k 15/17, 60 k 23/22
  //        128 -> 128 (tiles of 512 rows)      60 k 133/91 in boxes, 12 k 42/56; 128 -> 64 with one pair a row,
  //                                            150 k rows: 62/78
  //   row map, fp16 64 -> 64 150 k 1.2 times as fast, 30 k 0.9; 5x5x5 (whose map is read twice) 150 k 0.85
  double pairs = 0;
  for (int k = 0; k < p.K; ++k) pairs += (double)p.indice_num[k];
  const double fill = pairs / ((double)d.R * p.K);
  const double work = (double)d.R * (d.c_padded / 64);
  if (fill >= (p.K <= 8 ? 0.25 : 0.16)) return false;
  const bool long_rows = d.q_padded * (int)elemSize(p.dtype) > 256;
  if (lists) {
    if (tallHalfTiles(lc, p, d)) return true;
    if (long_rows) return work >= 85000 && pairs >= 1.1 * d.R;
    return p.K > kTallFewOffsets || work >= 45000;
  }
  return !long_rows && p.K <= 32 && d.q_padded >= 64 && work >= (d.c_padded == 128 ? 50000 : 80000);
}

// Shapes of gatherConvDenseStaged that add up by offset.
constexpr bool denseByOffsetShape(int elem_bytes, int Q, int C) { return elem_bytes == 2 && Q >= 64 && C >= 64; }

// How the register-accumulating kernel adds up, if it is used: all products of a row in one chain, or each offset's by
// itself, as the pair-list kernels do.
enum class DenseSums { kNone, kChain, kByOffset };

DenseSums useDenseKernel(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d, bool lists) {
  if (!denseShapeOk(p, d) || lc.choices.dense_tiles == 0) return DenseSums::kNone;
  // What the kernel costs goes with the (tile, offset) pieces that hold a pair at all, what
  // the pair-list kernels cost with the pairs.  Measured on 150000 rows, 3x3x3, as the share of all
  // (row, offset) slots that hold a pair from which the kernel wins, with us of the pair-list kernels
  // against us of this one around it:
  //   reduction -> result channels     voxels strewn uniformly               scenes (filled sheets and walls)
  //   fp16   16 -> 16                  0.18 (0.15: 24/26, 0.27: 31/26)       0.045 (0.04: 18/19, 0.05: 23/19)
  //          32 -> 32                  0.18 (0.15: 28/31, 0.27: 36/30)       0.045 (0.04: 20/21, 0.05: 27/20)
  //          16, 32 -> 64              0.14 (0.13: 39/41, 0.18: 47/41)       0.06  (0.05: 31/29, 0.10: 46/32)
  // Rows of 2-byte types above 64 bytes, since they go through LDS, are ahead around 0.2 strewn; the lines stayed, so that no
  // layer's sums changed, and below them each offset's product goes by itself (see below):
  //          64 -> 64                  0.27 (0.26: 69/56, 0.31: 77/57)      0.085 (0.18: 50/46, 0.26: 74/54, 0.35: 121/72)
  //          64 -> 128                 0.27 (0.26: 102/87, 0.31: 118/81)    0.05  (0.18: 77/59, 0.26: 109/72, 0.35: 178/96)
  //          128 -> 64                 0.27 (0.26: 98/86, 0.31: 111/87)     0.085 (0.18: 70/70, 0.26: 109/80, 0.35: 187/110)
  //          128 -> 128                0.27 (0.26: 149/131, 0.31: 170/133)  0.05  (0.18: 108/92, 0.26: 159/115, 0.35: 258/160)
  // The line of 64 result columns on scenes dates from pair-list kernels without tall tiles, which are ahead of this one
  // up to 0.16 filled (64 -> 64) and 0.18 (128 -> 64): thinned scenes, us of those / this,
  //   64 -> 64    5 k rows 0.09 20/26  0.14 23/27  0.18 27/27    20 k 0.12 22/27  0.17 28/27  0.24 33/27
  //               45 k 0.08 25/30  0.15 33/30    100 k 0.09 25/30  0.12 37/34  0.145 41/45  0.18 51/45
  //   128 -> 64   5 k 0.09 22/37  0.18 35/37  0.24 44/39    20 k 0.12 25/36  0.19 38/35    45 k 0.15 39/40  0.20 44/42
  //               100 k 0.145 51/65  0.18 69/66  0.26 87/65
  //   fp32   16 -> 16, 32              0.3  (0.22: 46/54, 0.4: 66/54)        0.05  (0.04: 26/31, 0.07: 49/38)
  //          32 -> 32                  0.4  (0.31: 81/95, 0.5: 114/95)       0.065 (0.05: 46/57, 0.10: 95/72)
  //          32 -> 64                  0.5  (0.4: 138/160, 0.5: 160/159)     0.15  (0.11: 111/125, 0.17: 138/129)
  //          64 -> 64                  -    (0.5: 275/338)                   0.2   (0.17: 231/242, 0.27: 294/245)
  //          64 -> 128                 -    (0.5: 485/636)                   -     (0.27: 462/450, 0.33: 471/505)
  // On strewn voxels every piece holds a few pairs; in a scene the pairs of an offset sit in
  // few pieces.  The host only knows the pair counts: sheets and walls show there as offsets
  // with far more pairs than the average offset (in-plane neighbours), which strewn voxels
  // never have.
  double pairs = 0, largest = 0, second = 0;
  for (int k = 0; k < p.K; ++k) {
    const double n = (double)p.indice_num[k];
    pairs += n;
    if (n > largest) {
      second = largest;
      largest = n;
    } else if (n > second) {
      second = n;
    }
  }
  const double fill = pairs / ((double)d.R * p.K);
  // (the largest count is the centre offset of a submanifold convolution: left out)
  const double mean_rest = p.K > 1 ? (pairs - largest) / (p.K - 1) : 0.0;
  const bool sheets = mean_rest > 0 && second >= 1.5 * mean_rest;
  bool chain;
  if (p.dtype != ElemType::kFloat) {
    chain = fill >= (sheets ? (d.q_padded >= 64 && d.c_padded == 64 ? 0.085 : 0.05) : (d.q_padded <= 32 ? 0.17 : 0.27));
  } else if (d.c_padded <= 32) {
    chain = fill >= (sheets ? 0.06 : 0.35);
  } else if (d.c_padded == 64) {
    chain = fill >= (sheets ? 0.18 : 0.5);
  } else {
    chain = sheets && d.q_padded <= 32 && fill >= 0.2;
  }
  // Fewer pairs, 2-byte rows of more than 64 bytes: with each offset's product by itself, which gives the pair-list
  // kernels' bits, so that a layer's results do not depend on this line.  It pays where some tiles hold far more pairs
  // than others: filled sheets, which show less in a strided layer's counts.  Strewn voxels differ in theirs as chance
  // has it, by some square roots of the count (1 500 rows: the second count 1.11 of the mean).  Up to 27 offsets: of 125, 5 k
  // strewn rows 64 -> 64 take 71/101.  us of the pair-list kernels / this one with the filter's packing, fp16, 3x3x3:
  //   stride 2 on scenes, 0.16 to 0.20 filled (second count 1.11 to 1.27 of the mean)
  //     64 -> 64    5 k rows 38/30   38 k 40/33   60 k 48/35   110 k 78/55   168 k 79/60
  //     128 -> 64   5 k 51/39   38 k 56/45   60 k 69/46   110 k 116/80
  //     64 -> 128   11 k 34/37   19 k 35/37   38 k 43/42   60 k 58/43   168 k 119/82
  //     128 -> 128  11 k 48/49   38 k 59/61   60 k 80/60   110 k 142/107        96 -> 96  38 k 58/62
  //   stride 2 on even walls and floors, 0.19 filled (1.17 to 1.35, by which the host cannot tell them from scenes; at
  //   0.23 filled the two are level from 2.5 k rows on)
  //     64 -> 64    0.8 k 25/29   2.5 k 27/29   7 k 28/30   28 k 30/31   51 k 34/33      128 -> 64   2.5 k 34/39   28 k 39/40   51 k 46/45
  //   strewn (1.02 to 1.39 at few rows), 64 -> 64 and 128 -> 64
  //     300 rows 0.18 24/30, 31/42   1 500 0.20 25/31, 31/42   16 k 0.21 26/31, 33/42   120 k 0.22 51/57, 70/82
  //   64 -> 128, strewn     50 k rows 0.18 41/44  0.22 44/44  0.25 47/44   120 k 0.18 70/73  0.21 74/75  0.25 81/76
  //                         160 k 0.18 87/82   250 k 0.18 136/121   16 k 0.21 25/37
  //   64 -> 128, stride 2 on what layers have thickened (1.02)    56 k 0.18 48/44   90 k 0.18 63/53   185 k 0.20 104/97
  //              2x2x2, stride 2 (1.00 to 1.03)    42 k 0.24 25/25   104 k 0.24 38/39   117 k 0.27 51/40   155 k 0.24 49/44
  const bool uneven = second >= 1.1 * mean_rest && second >= mean_rest + 4.0 * std::sqrt(mean_rest);
  const bool strided = largest < 0.9 * d.R;  // (a submanifold layer has every row in its centre)
  const double from = uneven ? (d.c_padded == 64 ? 1300 : d.q_padded == 64 ? 30000 : 50000) : p.K > 8 ? 50000 : 100000;
  const bool by_offset = !chain && lists && denseByOffsetShape((int)elemSize(p.dtype), d.q_padded, d.c_padded) &&
                         p.K <= 27 && fill >= 0.16 && d.R >= from &&
                         (uneven || (d.q_padded == 64 && d.c_padded == 128 && (strided || fill >= 0.22)));
  if (by_offset) return DenseSums::kByOffset;
  return chain || lc.choices.dense_tiles == 1 ? DenseSums::kChain : DenseSums::kNone;
}

// Pieces of a phase of gatherConvDenseStaged, 2-byte types: one or two.  Two halve the round trips that follow each other
// in a tile, and leave a CU two workgroups instead of three: for launches of few tiles, and for rows strewn over memory
// (`scattered`), whose two halves are then fetched together.  Row maps of 128 result columns take two always (their kernel
// needs the registers of two workgroups).  us with the filter's packing, one / two pieces, 3x3x3, 0.19 to 0.38 filled:
//   lists, rows in order    64 -> 16   1 k rows 24.9/22.2  20 k 23.0/21.6  120 k 40/39  250 k 65/69
//                           64 -> 32   1 k 25.5/23  20 k 23.6/23.5  50 k 26.0/27.0
//                           128 -> 32  1 k 37/31.5  20 k 31/31  50 k 39/36  120 k 63/61  250 k 100/106
//                           64 -> 64   1 k 27.4/25.4  8 k 26.7/25.8  20 k 26.5/26.4  50 k 30.4/30.7  250 k 75/84
//                           128 -> 64  1 k 39/35  8 k 37.7/35.8  20 k 35.6/36.9  50 k 43/44  250 k 112/126
//                           128 -> 128 1 k 45/43  8 k 43.9/45.4  250 k 157/171
//   lists, rows in no order 64 -> 16   1 k 26/23  20 k 26/23  120 k 56/48  300 k 107/104     64 -> 64  1 k 28/26  20 k 29/27
//                           120 k 59/56  300 k 115/120     128 -> 64  20 k 42/38  120 k 94/88  300 k 190/193
//   row maps, no order      64 -> 64   8 k 41/37  120 k 90/85  300 k 161/162   128 -> 128  20 k 71/59  120 k 170/150  300 k 358/322
//   row maps, rows in order 64 -> 64   1 k 25/23  20 k 24.5/24.4  300 k 78/88   128 -> 128  20 k 47/45  300 k 223/204
int denseDepth(bool lists, bool scattered, int q_padded, int c_padded, int rows) {
  if (c_padded == 128) return lists ? 1 : 2;
  if (scattered) return !lists || c_padded <= 32 || rows <= 131072 ? 2 : 1;
  if (c_padded == 64) return rows <= (q_padded == 64 ? 32768 : 10000) ? 2 : 1;
  return rows <= (q_padded == 64 && c_padded == 32 ? 32768 : 131072) ? 2 : 1;
}

template <typename E, int Q, int C, typename SRC>
void launchDenseInstance(const LaunchCtx &lc, const void *A, uint32_t a_size, const ConvRows &rows,
                         const void *packed, const SRC &source, bool by_offset, bool scattered, int R, int K,
                         void *result) {
  auto launch = [&](auto kernel) {
    lc.begin(by_offset ? "gatherConvDenseByOffset" : "gatherConvDense");
    kernel<<<denseGridX(R), kDenseThreads, 0, lc.stream>>>(
        static_cast<const typename E::storage *>(A), a_size, rows, static_cast<const typename E::storage *>(packed),
        source, R, K, static_cast<typename E::storage *>(result));
    lc.end();
  };
  if constexpr (SRC::kSegments && denseByOffsetShape((int)sizeof(typename E::storage), Q, C)) {
    if (by_offset) return launch(gatherConvDenseStaged<E, Q, C, true, 1, SRC>);
  }
  if constexpr (Q * (int)sizeof(typename E::storage) > 64) {
    if constexpr (sizeof(typename E::storage) == 2 && !(SRC::kSegments && C == 128)) {
      if (C == 128 || denseDepth(SRC::kSegments, scattered, Q, C, R) == 2)
        return launch(gatherConvDenseStaged<E, Q, C, false, 2, SRC>);
    }
    if constexpr (sizeof(typename E::storage) == 4 || SRC::kSegments || C < 128)
      launch(gatherConvDenseStaged<E, Q, C, false, 1, SRC>);
  } else {
    launch(gatherConvDense<E, Q, C, SRC>);
  }
}

template <typename E, typename SRC>
void launchDense(const LaunchCtx &lc, int q_padded, const void *A, int n_src, const ConvRows &rows,
                 const void *packed, const SRC &source, bool by_offset, bool scattered, int R, int K, void *result) {
  const uint32_t a_size = (uint32_t)n_src * (uint32_t)rows.row_bytes;
#define DENSE_INSTANCE(q, c) launchDenseInstance<E, q, c, SRC>(lc, A, a_size, rows, packed, source, by_offset, scattered, R, K, result)
#define DENSE_BY_C(q)                       \
  switch (rows.c_padded) {                  \
    case 16: DENSE_INSTANCE(q, 16); break;  \
    case 32: DENSE_INSTANCE(q, 32); break;  \
    case 64: DENSE_INSTANCE(q, 64); break;  \
    default: DENSE_INSTANCE(q, 128); break; \
  }
  switch (q_padded) {
    case 16: DENSE_BY_C(16) break;
    case 32: DENSE_BY_C(32) break;
    case 64: DENSE_BY_C(64) break;
    case 128:
      if constexpr (!std::is_same<E, FloatElem>::value) { DENSE_BY_C(128) }
      break;
    default: break;
  }
#undef DENSE_BY_C
#undef DENSE_INSTANCE
}

template <typename E, int Q, int C>
void launchSingleInstance(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d, const OffsetCounts &inl,
                          const void *A, const ConvRows &rows, const void *packed, void *result) {
  constexpr int RB = Q * (int)sizeof(typename E::storage) < 64 ? 64 : Q * (int)sizeof(typename E::storage);
  OffsetBlocks ob;
  int blocks = 0;
  for (int k = 0; k < kMaxInlineK; ++k) {
    ob.first[k] = blocks;
    if (k < p.K) blocks += (inl.n[k] + singlePairs(RB) - 1) / singlePairs(RB);
  }
  if (blocks == 0) return;
  lc.begin("gatherConvSingle");
  gatherConvSingle<E, Q, C><<<blocks, kDenseThreads, 0, lc.stream>>>(
      static_cast<const typename E::storage *>(A), (uint32_t)d.n_src * (uint32_t)rows.row_bytes, rows,
      static_cast<const typename E::storage *>(packed), p.indice_pairs, p.L, d.row_col, d.src_col, inl, ob, p.K, d.R,
      d.n_src, static_cast<typename E::storage *>(result));
  lc.end();
}

template <typename E>
void launchSingle(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d, const OffsetCounts &inl, const void *A,
                  const ConvRows &rows, const void *packed, void *result) {
#define SINGLE_INSTANCE(q, c) launchSingleInstance<E, q, c>(lc, p, d, inl, A, rows, packed, result)
#define SINGLE_BY_C(q)                       \
  switch (d.c_padded) {                      \
    case 16: SINGLE_INSTANCE(q, 16); break;  \
    case 32: SINGLE_INSTANCE(q, 32); break;  \
    case 64: SINGLE_INSTANCE(q, 64); break;  \
    default: SINGLE_INSTANCE(q, 128); break; \
  }
  switch (d.q_padded) {
    case 16: SINGLE_BY_C(16) break;
    case 32: SINGLE_BY_C(32) break;
    case 64: SINGLE_BY_C(64) break;
    default: SINGLE_BY_C(128) break;
  }
#undef SINGLE_BY_C
#undef SINGLE_INSTANCE
}

// Row maps are built on the flat grid from this many workgroups of the per-offset grid on.
constexpr int kFlatScatterFromBlocks = 16384;

// Caller brackets this with its timing marks.  dev_counts != nullptr: more offsets
// than the inline tables hold, counts in device memory, grid kernel only.  Returns the
// number of workgroups, each of which writes one entry of `accepted`.
int enqueueScatterRowMap(const LaunchCtx &lc, const int32_t *pairs, int L, int K,
                         const OffsetCounts &inl, const int32_t *dev_counts, int max_count,
                         int row_col, int src_col, int row_base, int n_rows, int n_src,
                         int32_t *map, int32_t *accepted, RunIf run_if) {
  const int gx = (max_count + 255) / 256 > 1024 ? 1024 : (max_count + 255) / 256;
  if (dev_counts == nullptr && K <= kMaxInlineK &&
      (lc.choices.flat_scatter == 1 ||
       (lc.choices.flat_scatter != 0 && (long long)gx * K > kFlatScatterFromBlocks))) {
    OffsetBlocks ob;
    int blocks = 0;
    for (int k = 0; k < K; ++k) {
      ob.first[k] = blocks;
      blocks += inl.n[k] > 0 ? (inl.n[k] + 255) / 256 : 0;
    }
    if (blocks > 0)
      scatterRowMapFlat<<<blocks, 256, 0, lc.stream>>>(pairs, L, inl, ob, K, row_col, src_col,
                                                   row_base, n_rows, n_src, map, accepted, run_if);
    return blocks;
  }
  scatterRowMap<<<dim3(gx, K), 256, 0, lc.stream>>>(pairs, L, inl, dev_counts, row_col, src_col,
                                                 row_base, n_rows, n_src, map, accepted, run_if);
  return gx * K;
}

// The map of result rows [row_base, row_base + n_rows); returns the entries of ws.accepted written.
int launchScatterRowMap(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d,
                        const GatherWorkspace &ws, const OffsetCounts &inl, int max_count,
                        int row_base, int n_rows, RunIf run_if) {
  if (max_count <= 0) return 0;
  lc.begin("scatterRowMap");
  const int n = enqueueScatterRowMap(lc, p.indice_pairs, p.L, p.K, inl, ws.dev_counts, max_count,
                                     d.row_col, d.src_col, row_base, n_rows, d.n_src, ws.map, ws.accepted,
                                     run_if);
  lc.end();
  return n;
}

template <typename E>
void launchGatherTyped(const LaunchCtx &lc, const ConvProblem &p, const GatherDims &d,
                       const GatherWorkspace &ws, const OffsetCounts &inl, int max_count,
                       const void *gathered, const FilterView &f, bool use_mfma, void *result) {
  typedef typename E::storage S;
  // B(k, q, c): forward q = ci, c = co; backward data q = co, c = ci.
  const int64_t sQ = d.filter_forward ? f.stride_ci : f.stride_co;
  const int64_t sC = d.filter_forward ? f.stride_co : f.stride_ci;
  const int chunks = (d.q_padded + E::kChunk - 1) / E::kChunk, groups = d.c_padded / 16;
  FilterShape shape = {d.Q, d.C, 0, 0, d.Q == chunks * E::kChunk && d.C == d.c_padded};
  while (1 << shape.chunk_bits < chunks) ++shape.chunk_bits;
  while (1 << shape.group_bits < groups) ++shape.group_bits;
  const bool pad_rows = use_mfma && rowsNeedPadding(p.dtype, d.Q);
  const ConvRows rows_of = {d.Q, pad_rows ? paddedRowBytes(p.dtype, d.Q) : d.Q * (int)sizeof(S), d.C, d.c_padded, p.relu};
  const void *rows_from = pad_rows ? ws.padded_rows : gathered;
  const PadRows pad = {static_cast<const char *>(gathered), static_cast<char *>(ws.padded_rows), d.Q * (int)sizeof(S),
                       rows_of.row_bytes, pad_rows ? d.n_src : 0, pad_rows ? gridFor((size_t)d.n_src, 1024) : 0};
  const size_t frags = (size_t)p.K * groups * chunks * 64;
  if (p.single_pairs && use_mfma && p.row_map == nullptr && p.K <= kMaxInlineK &&
      (uint64_t)d.n_src * (uint64_t)rows_of.row_bytes < (uint64_t)kNoRow) {
    int64_t pairs = 0;
    for (int k = 0; k < p.K; ++k) pairs += inl.n[k];
    const size_t elems = pairs < d.R ? (size_t)d.R * d.C : 0;  // to be cleared: some rows are in no pair
    const int fill_blocks = elems > 0 ? gridFor(elems * sizeof(S) / 16 + 1, 2048) : 0;
    lc.begin("clearResultPackFilter");
    clearResultPackFilter<E><<<pad.blocks + fill_blocks + gridFor(frags, 512), 256, 0, lc.stream>>>(
        pad, static_cast<S *>(result), elems, fill_blocks, static_cast<const S *>(f.base), f.stride_k, sQ, sC, p.K, shape,
        static_cast<S *>(ws.packed), p.ticket);
    lc.end();
    launchSingle<E>(lc, p, d, inl, rows_from, rows_of, ws.packed, result);
    return;
  }
  const bool single_chunk = p.row_map == nullptr && ws.map_rows >= d.R && lc.choices.small_map_chunks != 1;
  // Pair lists whose order nobody has reported yet: the call starts on them all the same,
  // and the row-map kernels are enqueued behind, each of them told to return at once unless
  // the first kernel found the lists out of order (then the list kernel returns at once
  // instead).  Worth it only where the row map is a single chunk of four launches.
  const bool speculate = p.list_trust == ListTrust::kUnknown && single_chunk && lc.choices.lists_on_trust != 0;
  const bool lists = use_mfma && listsUsable(p, d) && (p.list_trust == ListTrust::kInOrder || speculate);
  const DenseSums dense_sums = use_mfma ? useDenseKernel(lc, p, d, lists) : DenseSums::kNone;
  const bool dense = dense_sums != DenseSums::kNone;
  const bool tall = use_mfma && !dense && useTallKernel(lc, p, d, lists);
  const int tall_q = tallQ(p.dtype, d.q_padded);
  const int tall_rows = tall ? tallTileRows(lc, p, d, tall_q, lists) : 0;
  if (lists) {
    // Pair lists in order (as far as the caller knows: the first kernel checks): the
    // gather kernel reads them cut by tile, no row map.
    const int tile_cols = dense ? d.c_padded : mfmaTileCols(p, d);
    const int tile_rows = dense ? kDenseRows : tall ? tall_rows : mfmaTileRows(tile_cols);
    int tile_shift = 0;
    while ((1 << tile_shift) < tile_rows) ++tile_shift;
    const int n_tiles = (d.R + tile_rows - 1) / tile_rows;
    OffsetBlocks ob;
    int list_blocks = 0;
    for (int k = 0; k < kMaxInlineK; ++k) {
      ob.first[k] = list_blocks;
      const int per_block = 256 * kCutPairsPerThread;
      if (k < p.K) list_blocks += inl.n[k] > 0 ? (inl.n[k] + per_block - 1) / per_block : 1;
    }
    const int pack_blocks = gridFor(frags, 512);
    lc.begin("packFilterCutPairLists");
    packFilterCutPairLists<E><<<pad.blocks + pack_blocks + list_blocks, 256, 0, lc.stream>>>(
        pad, static_cast<const S *>(f.base), f.stride_k, sQ, sC, p.K, shape, static_cast<S *>(ws.packed),
        pack_blocks, p.indice_pairs, p.L, inl, ob, d.row_col, d.src_col, d.R, d.n_src, tile_shift,
        n_tiles, ws.cuts, ws.verdict, p.ticket);
    lc.end();
    SegmentSource src;
    src.pairs = p.indice_pairs;
    src.cuts = ws.cuts;
    src.verdict = ws.verdict;
    src.ticket = p.ticket;
    src.leave_if_unordered = speculate;
    src.L = p.L;
    src.row_col = d.row_col;
    src.src_col = d.src_col;
    src.n_src = d.n_src;
    src.cut_stride = n_tiles + 1;
    src.W = f.base;
    src.sK = f.stride_k;
    src.sQ = sQ;
    src.sC = sC;
    src.counts = inl;
    if (dense)
      launchDense<E, SegmentSource>(lc, d.q_padded, rows_from, d.n_src, rows_of, ws.packed, src,
                                    dense_sums == DenseSums::kByOffset, p.scattered, d.R, p.K, result);
    else if (tall)
      launchTall<E, SegmentSource>(lc, tall_q, rows_from, d.n_src, rows_of, ws.packed, src, tall_rows, d.R, p.K,
                                   result);
    else if (tile_cols == d.c_padded && useWaveKernel(lc, p.dtype, d.q_padded, d.c_padded))
      launchWave<E>(lc, d.q_padded, rows_from, rows_of, ws.packed, src, d.R, p.K, result);
    else
      launchMfma<E, SegmentSource>(lc, d.q_padded, tile_cols, rows_from, rows_of, ws.packed, src, d.R, p.K, result);
    if (!speculate || lc.choices.lists_on_trust == 1) return;
  }
  // What follows runs always, or (behind lists taken on trust) only when they failed the check.
  const RunIf run_if = lists ? RunIf{ws.verdict, p.ticket} : RunIf{nullptr, 0};
  const bool own_map = p.row_map == nullptr;  // else: built ahead, nothing to clear or fill
  // A map of the library's own covers a chunk of result rows at a time: filled, used by the
  // gather kernel for those rows, checked for lost pairs, and filled again for the next rows.
  int chunk_rows = own_map ? ws.map_rows : d.R;
  if (own_map && lc.choices.small_map_chunks == 1 && chunk_rows > kRepairPoolRows) chunk_rows = kRepairPoolRows;
  // (what goes by pair lists only: sums by offset, and tall tiles of another height than the row maps')
  const bool map_dense = dense_sums == DenseSums::kChain;
  const int map_tall_rows = tallRows(tall_q * (int)sizeof(S));
  const int tile_cols = use_mfma && !map_dense ? mfmaTileCols(p, d) : d.c_padded;
  for (int row_base = 0; row_base < d.R; row_base += chunk_rows) {
    const int rows = d.R - row_base < chunk_rows ? d.R - row_base : chunk_rows;
    const size_t map_elems = (size_t)p.K * rows;
    const int32_t *entries = own_map ? ws.map : p.row_map;
    S *result_rows = static_cast<S *>(result) + (size_t)row_base * d.C;
    int n_filled = 0;    // workgroups along x of the gather kernel = slot counts it leaves
    int n_accepted = 0;  // workgroups of the map scatter = counts of pairs it leaves
    if (use_mfma) {
      // the filter is repacked with the first chunk's map fill (the list kernels' first
      // launch has done it already where they ran)
      const int fill_blocks = own_map ? gridFor(map_elems / 4 + 1, 2048) : 0;
      const int pack_blocks = row_base == 0 && !lists ? gridFor(frags, 512) : 0;
      PadRows pad_now = pad;
      if (pack_blocks == 0) pad_now.blocks = 0;
      if (fill_blocks + pack_blocks > 0) {
        lc.begin("fillMapPackFilter");
        fillMapPackFilter<E><<<pad_now.blocks + fill_blocks + pack_blocks, 256, 0, lc.stream>>>(
            pad_now, ws.map, map_elems, fill_blocks, static_cast<const S *>(f.base), f.stride_k, sQ, sC, p.K,
            shape, static_cast<S *>(ws.packed), p.ticket, run_if);
        lc.end();
      }
      if (own_map) n_accepted = launchScatterRowMap(lc, p, d, ws, inl, max_count, row_base, rows, run_if);
      const MapSource map = {entries, ws.filled, run_if};
      if (map_dense) {
        n_filled = denseGridX(rows);
        launchDense<E, MapSource>(lc, d.q_padded, rows_from, d.n_src, rows_of, ws.packed, map, false,
                                  p.list_trust != ListTrust::kInOrder || p.scattered, rows, p.K, result_rows);
      } else if (tall) {
        n_filled = tallGridX(rows, map_tall_rows);
        launchTall<E, MapSource>(lc, tall_q, rows_from, d.n_src, rows_of, ws.packed, map, map_tall_rows, rows, p.K,
                                 result_rows);
      } else {
        n_filled = mfmaGridX(rows, tile_cols);
        launchMfma<E, MapSource>(lc, d.q_padded, tile_cols, rows_from, rows_of, ws.packed, map, rows, p.K, result_rows);
      }
    } else {
      if (own_map) {
        lc.begin("fillInt32");
        fillInt32<<<gridFor(map_elems), 256, 0, lc.stream>>>(ws.map, map_elems, -1);
        lc.end();
        n_accepted = launchScatterRowMap(lc, p, d, ws, inl, max_count, row_base, rows, run_if);
      }
      dim3 grid((rows + 31) / 32, (d.C + 63) / 64);
      n_filled = (int)grid.x;
      lc.begin("gatherConvSimt");
      gatherConvSimt<E><<<grid, 256, 0, lc.stream>>>(static_cast<const S *>(gathered), d.Q,
                                                  static_cast<const S *>(f.base), f.stride_k, sQ, sC,
                                                  entries, rows, p.K, inl, ws.dev_counts, d.C,
                                                  ws.filled, p.relu, result_rows);
      lc.end();
    }
    if (p.distinct_pairs || !own_map) continue;  // a map built ahead was checked when it was built
    // returns at once unless pairs of one offset share a result row
    lc.begin("repairLostPairs");
    repairLostPairs<E><<<repairBlocks(rows), 256, 0, lc.stream>>>(
        static_cast<const S *>(gathered), d.Q, static_cast<const S *>(f.base), f.stride_k, sQ, sC,
        p.indice_pairs, p.L, d.row_col, d.src_col, rows, d.n_src, p.K, row_base, inl, ws.dev_counts,
        ws.map, ws.filled, n_filled, ws.accepted, n_accepted, d.C,
        RepairScratch{ws.shadow, ws.pool_row, ws.pool}, p.relu, result_rows, run_if);
    lc.end();
  }
}

struct FilterGradWorkspace {
  int32_t *dev_counts = nullptr;
  float *partial = nullptr;
  int splits = 1;
  size_t bytes = 0;
};

bool filterMfmaShapeOk(const ConvProblem &p) {
  return mfmaShapeOk(p.Ci, p.Co) && p.K <= kMaxInlineK;
}

// Slices the MFMA kernels cut the pair lists into at most: kFilterMaxSlices (fewer for many
// offsets), or what a capped workspace leaves beside one tile per offset.
int filterMaxSlices(const ConvProblem &p) {
  const int most = p.K <= kFilterFewOffsets ? kFilterMaxSlices : kFilterMaxSlicesManyOffsets;
  if (p.max_partial_tiles <= 0) return most;
  const int room = p.max_partial_tiles - p.K;
  return room < 1 ? 1 : (room > most ? most : room);
}

int filterGradSplits(const ConvProblem &p) {
  // Bounded by the tensor shape only, so the workspace query and the launch
  // agree whatever indice_num holds.
  int s = (p.L + 4095) / 4096;
  if (s < 1) s = 1;
  if (s > 32) s = 32;
  return s;
}

FilterGradWorkspace carveFilterGrad(const ConvProblem &p, void *base) {
  FilterGradWorkspace ws;
  char *ptr = alignPtr(base);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *r = ptr ? ptr + off : nullptr;
    off += alignUp(bytes);
    return r;
  };
  if (p.K > kMaxInlineK) ws.dev_counts = reinterpret_cast<int32_t *>(take((size_t)p.K * 4));
  ws.splits = filterGradSplits(p);
  size_t elems = ws.splits > 1 ? (size_t)ws.splits * p.K * p.Ci * p.Co : 0;
  // the MFMA path writes at most filterMaxSlices + K partial tiles of padded channels
  if (filterMfmaShapeOk(p)) {
    const size_t tiles = (size_t)filterMaxSlices(p) + p.K;
    const size_t mfma_elems = tiles * paddedChannels(p.Ci) * paddedChannels(p.Co);
    if (mfma_elems > elems) elems = mfma_elems;
  }
  if (elems > 0) ws.partial = reinterpret_cast<float *>(take(elems * 4));
  ws.bytes = off + kBaseAlign;
  return ws;
}

// filters_grad is [K, Ci, Co] unless the caller asked for another layout.
GradLayout gradLayout(const ConvProblem &p) {
  GradLayout g;
  if (p.grad_stride_k == 0 && p.grad_stride_ci == 0 && p.grad_stride_co == 0) {
    g.stride_k = (int64_t)p.Ci * p.Co; g.stride_ci = p.Co; g.stride_co = 1;
  } else {
    g.stride_k = p.grad_stride_k; g.stride_ci = p.grad_stride_ci; g.stride_co = p.grad_stride_co;
  }
  return g;
}

// Rows that the backward filter reads into LDS as they are: 2-byte operands are transposed by LDS reads, fp32 ones need
// no transposition.
bool transposingReads(const LaunchCtx &lc, const ConvProblem &p) {
  // (rows are addressed with 32-bit byte offsets; the API's tensors have less than 2^31 elements)
  const uint64_t x_bytes = (uint64_t)(p.inverse ? p.num_out : p.L) * (uint64_t)p.Ci * elemSize(p.dtype);
  const uint64_t y_bytes = (uint64_t)(p.inverse ? p.L : p.num_out) * (uint64_t)p.Co * elemSize(p.dtype);
  return p.Ci > 16 && p.Co > 16 && lc.choices.filter_stores != 1 && !rowsNeedPadding(p.dtype, p.Ci) &&
         !rowsNeedPadding(p.dtype, p.Co) && x_bytes <= kNoPlace && y_bytes <= kNoPlace;
}

// Workgroups of the walks (walkOfWorkgroup), 0: slices.  As many as are resident at a time, so that all
// of them are at about the same rows: 512 at 128 x 128 channels, 768 with 128 on one side, and from 1.5 M
// pairs on, where a second round no longer shows, 1024.  Fewer pairs leave walks of a few steps.  us with the
// sums, slices against walks of 512 / 768 / 1024 workgroups, scenes, 3x3x3, fp16:
//   128 x 128   0.50 M pairs 44/44/-/54   0.72 M 69/64/-/70   2.0 M 129/103/-/110   2.85 M 180/145/-/146
//    96 x 96    1.6 M 118/100/108/95      3.0 M 205/163/174/148
//    64 x 128   0.57 M 36/36/36/39        0.78 M 53/43/41/46  2.0 M 87/109/79/74    3.0 M 111/159/110/94
//    64 x 64    0.50 M 26/27/-/25         0.84 M 36/38/-/36   1.05 M 36/41/-/33     2.0 M 66/94/-/56
//    32 x 32    0.50 M 20/22/-/19         0.84 M 28/31/-/25   2.0 M 56/76/-/45
int filterWalkers(const ConvProblem &p, long long pairs) {
  if (p.K > kFilterFewOffsets) return 0;
  const int channels = paddedChannels(p.Ci) + paddedChannels(p.Co);
  if (pairs < (channels == 256 ? 600000 : (channels >= 192 ? 700000 : 800000))) return 0;
  int want = kFilterMaxSlices;
  if (pairs < 1500000 && channels >= 192) want = channels == 256 ? 512 : 768;
  if (want > filterMaxSlices(p)) want = filterMaxSlices(p);  // (a capped workspace)
  return want / kFilterShares < p.K ? 0 : want;
}

template <typename E, int CI, int CO>
void launchFilterMfmaInstance(const LaunchCtx &lc, const ConvProblem &p, const SliceTable &tab,
                              const SliceOrder &order, int slice_len, int shares, int total_slices, float *partial,
                              const void *features, const void *output_grad, void *filters_grad) {
  typedef typename E::storage S;
  constexpr bool kTransposingShape = CI >= 32 && CO >= 32;
  const bool transposing = kTransposingShape && transposingReads(lc, p);
  const FilterGradRows rows = {p.Ci, p.Co};
  const int grid = shares > 0 ? shares * total_slices : (total_slices + 7) / 8 * 8;
  lc.begin(!transposing ? "backwardFilterMfma" : (sizeof(S) == 4 ? "backwardFilterMfmaRows" : "backwardFilterMfmaTr"));
  if (total_slices > 0) {
    const bool whole = p.Ci == CI && p.Co == CO;
    auto kernel = backwardFilterMfma<E, CI, CO, false>;
    if constexpr (!kTransposingShape) {
      if (whole) kernel = backwardFilterMfma<E, CI, CO, true>;
    }
    if constexpr (kTransposingShape) {
      // fp32 takes steps of 32 pairs, 2-byte types of 64, half as many barriers; with 128 channels on a side those
      // leave two or three workgroups' buffers on a CU, and where a workgroup has many steps the shorter ones, with
      // four, are faster (in walks: slices of 125 offsets, 1.6 M pairs, 128 x 128, 141/131).  us with the sums, fp16,
      // steps of 32 / 64:
      //   3.0 M pairs   32 x 32 55/39   32 x 64 62/50   64 x 64 67/57   32 x 128 73/83   64 x 128 89/100   128 x 128 135/142
      //   0.98 M pairs  32 x 32 28/23   64 x 64 35/31   64 x 128 43/41   128 x 128 67/59;  fp32  64 x 64 86/98   128 x 128 302/317
      auto tr = backwardFilterRows<E, CI, CO, 32, false>;
      if (whole) tr = backwardFilterRows<E, CI, CO, 32, true>;
      if constexpr (sizeof(S) == 2) {
        const bool short_steps = (CI == 128 || CO == 128) && shares > 0 && slice_len >= 2048;
        if (!short_steps) tr = whole ? backwardFilterRows<E, CI, CO, 64, true> : backwardFilterRows<E, CI, CO, 64, false>;
      }
      if (transposing)
        tr<<<grid, 256, 0, lc.stream>>>(
            static_cast<const S *>(features), static_cast<const S *>(output_grad), rows, p.indice_pairs, p.L,
            p.inverse ? 1 : 0, p.inverse ? p.num_out : p.L, p.inverse ? p.L : p.num_out, p.K, tab, order,
            total_slices, slice_len, shares, partial);
    }
    if (!transposing)
      kernel<<<grid, 256, 0, lc.stream>>>(
          static_cast<const S *>(features), static_cast<const S *>(output_grad), rows, p.indice_pairs, p.L,
          p.inverse ? 1 : 0, p.inverse ? p.num_out : p.L, p.inverse ? p.L : p.num_out, p.K, tab, order,
          total_slices, slice_len, shares, partial);
  }
  lc.end();
  // Many offsets of few slices each: the flat grid, on which such an offset takes a
  // sixteenth of the workgroups (same bits).
  constexpr int kChunks = CI * CO / 256;
  SumGrid sg;
  int blocks = 0;
  for (int k = 0; k < p.K; ++k) {
    const int sl = tab.tiles[k];
    sg.first[k] = blocks;
    blocks += sl <= kThinSlices ? (kChunks + kSliceSumWaves - 1) / kSliceSumWaves : kChunks;
  }
  const int flat_mode = lc.choices.flat_slice_sum;
  const bool flat = flat_mode == 1 || (flat_mode < 0 && kChunks * p.K > kFlatSumFromBlocks);
  lc.begin("sliceSum");
  if (flat)
    sliceSumFlat<E><<<blocks, 64 * kSliceSumWaves, 0, lc.stream>>>(
        partial, tab, sg, p.K, slice_len, CI * CO, CO, rows, gradLayout(p), static_cast<S *>(filters_grad));
  else
    sliceSum<E><<<dim3(kChunks, p.K), 64 * kSliceSumWaves, 0, lc.stream>>>(
        partial, tab, slice_len, CI * CO, CO, rows, gradLayout(p), static_cast<S *>(filters_grad));
  lc.end();
}

template <typename E, int CI>
void launchFilterMfmaByCo(const LaunchCtx &lc, const ConvProblem &p, const SliceTable &tab,
                          const SliceOrder &order, int slice_len, int shares, int total_slices, float *partial,
                          const void *features, const void *output_grad, void *filters_grad) {
#define FILTER_INSTANCE(co)                                                                                        \
  case co:                                                                                                         \
    launchFilterMfmaInstance<E, CI, co>(lc, p, tab, order, slice_len, shares, total_slices, partial, features,     \
                                        output_grad, filters_grad);                                                \
    break;
  switch (paddedChannels(p.Co)) {
    FILTER_INSTANCE(16)
    FILTER_INSTANCE(32)
    FILTER_INSTANCE(64)
    FILTER_INSTANCE(128)
    default: break;
  }
#undef FILTER_INSTANCE
}

// Slice length from the real pair count: about kFilterMaxSlices workgroups
// whatever the density, and never more than kFilterMaxSlices + K partial tiles.
template <typename E>
void launchFilterMfma(const LaunchCtx &lc, const ConvProblem &p, const FilterGradWorkspace &ws,
                      const OffsetCounts &inl, const void *features, const void *output_grad,
                      void *filters_grad) {
  {
    SliceTable tab;
    long long total = 0;
    for (int k = 0; k < p.K; ++k) total += inl.n[k];
    // (the larger number of slices only where they stay long: a fourth workgroup a CU does not
    // fit, and a second round of short slices costs more than it spreads; config 3, 404 000
    // pairs: 24 us at 701 slices, 31 us at 789)
    int max_slices = filterMaxSlices(p);
    if (total < (long long)kFilterMaxSlices * 2048 && max_slices > kFilterMaxSlicesManyOffsets)
      max_slices = kFilterMaxSlicesManyOffsets;
    int slice_len = (int)((total + max_slices - 1) / max_slices);
    slice_len = (slice_len + kFilterStepPairs - 1) / kFilterStepPairs * kFilterStepPairs;
    // A slice has fixed costs (the first rows' round trip, a Ci x Co fp32 tile written and summed again), and a slice's
    // steps follow each other: few pairs are cut into about 192 slices and no finer than 256 pairs, nor, however many
    // the pairs are, finer than 1024 at 128 x 128 channels and 512 below, at the price of idle CUs.  fp32, whose
    // multiplies take eight times as long, is cut to 256 at once.  us with the sums, slices of 256 / 512 / 1024 pairs:
    //   fp16  128 x 128   20 000 pairs 22/24/29   91 000 32/29/31   277 000 41/42/37      64 x 64  20 000 14/15/18   91 000 17/16/18
    //   fp32  128 x 128   20 000 pairs 37/53/88   91 000 58/60/91   277 000 122/131/151   64 x 64  20 000 18/24/35   91 000 25/32/36
    const int most = paddedChannels(p.Ci) * paddedChannels(p.Co) >= 128 * 128 ? 1024 : 512;
    int least = 256;
    if (p.dtype != ElemType::kFloat) {
      const int spread = (int)((total + 191) / 192 < most ? (total + 191) / 192 : most);
      least = spread < 256 ? 256 : (spread + kFilterStepPairs - 1) / kFilterStepPairs * kFilterStepPairs;
    }
    if (slice_len < least) slice_len = least;
    // Walks instead of slices, and the workgroups an offset's share of its list is walked by: one each,
    // the others to the offsets whose walks are longest.
    int walkers[kMaxInlineK];
    const int per_share = filterWalkers(p, total) / kFilterShares;
    const int shares = per_share > 0 ? kFilterShares : 0;
    for (int k = 0; k < p.K; ++k) walkers[k] = inl.n[k] > 0 ? 1 : 0;
    for (int left = per_share - p.K; left > 0; --left) {
      int longest = 0;
      for (int k = 1; k < p.K; ++k)
        if ((long long)inl.n[k] * walkers[longest] > (long long)inl.n[longest] * walkers[k]) longest = k;
      ++walkers[longest];
    }
    int first = 0;
    for (int k = 0; k < kMaxInlineK; ++k) {
      const int n = k < p.K ? inl.n[k] : 0;
      tab.n[k] = n;
      tab.first[k] = first;
      tab.tiles[k] = shares == 0 ? (n + slice_len - 1) / slice_len : (k < p.K ? walkers[k] * shares : 0);
      first += tab.tiles[k];
    }
    const int entries = shares > 0 ? first / shares : first;
    SliceOrder order;
    int placed = 0;
    if (shares > 0) {
      // the longest walks of a share first
      int by_length[kMaxInlineK];
      for (int k = 0; k < p.K; ++k) by_length[k] = k;
      std::stable_sort(by_length, by_length + p.K, [&](int a, int b) {
        return (long long)inl.n[a] * walkers[b] > (long long)inl.n[b] * walkers[a];
      });
      for (int i = 0; i < p.K; ++i)
        for (int w = 0; w < walkers[by_length[i]]; ++w) order.offset[placed++] = (uint8_t)by_length[i];
    } else {
      // slices in the order of the share of their offset's list in front of them, in `steps`
      // steps of that share (as many as the longest list has slices)
      int steps = 1, next[kMaxInlineK];
      for (int k = 0; k < p.K; ++k) {
        next[k] = 0;
        if (tab.tiles[k] > steps) steps = tab.tiles[k];
      }
      for (int t = 0; t < steps; ++t)
        for (int k = 0; k < p.K; ++k)
          while (next[k] < tab.tiles[k] && (long long)next[k] * steps < (long long)(t + 1) * tab.tiles[k]) {
            order.offset[placed++] = (uint8_t)k;
            ++next[k];
          }
    }
#define FILTER_BY_CO(ci)                                                                                           \
  case ci:                                                                                                         \
    launchFilterMfmaByCo<E, ci>(lc, p, tab, order, slice_len, shares, entries, ws.partial, features, output_grad,  \
                                filters_grad);                                                                     \
    break;
    switch (paddedChannels(p.Ci)) {
      FILTER_BY_CO(16)
      FILTER_BY_CO(32)
      FILTER_BY_CO(64)
      FILTER_BY_CO(128)
      default: break;
    }
#undef FILTER_BY_CO
  }
}

template <typename E>
void launchFilterGradTyped(const LaunchCtx &lc, const ConvProblem &p,
                           const FilterGradWorkspace &ws, const OffsetCounts &inl,
                           const void *features, const void *output_grad, void *filters_grad) {
  typedef typename E::storage S;
  // The MFMA path moves rows with 16-byte loads.
  const bool ptr_ok = ((reinterpret_cast<uintptr_t>(features) |
                        reinterpret_cast<uintptr_t>(output_grad)) & 15u) == 0;
  if (filterMfmaShapeOk(p) && ptr_ok && lc.choices.gather_simt != 1) {
    launchFilterMfma<E>(lc, p, ws, inl, features, output_grad, filters_grad);
    return;
  }
  const int tiles = ((p.Ci + 31) / 32) * ((p.Co + 63) / 64);
  dim3 grid(tiles, p.K, ws.splits);
  lc.begin("backwardFilterSimt");
  backwardFilterSimt<E><<<grid, 256, 0, lc.stream>>>(
      static_cast<const S *>(features), static_cast<const S *>(output_grad), p.indice_pairs, p.L,
      p.inverse ? 1 : 0, p.inverse ? p.num_out : p.L, p.inverse ? p.L : p.num_out, p.Ci, p.Co, inl,
      ws.dev_counts, ws.splits, ws.partial, gradLayout(p), static_cast<S *>(filters_grad));
  lc.end();
  if (ws.splits > 1) {
    const size_t n = (size_t)p.K * p.Ci * p.Co;
    lc.begin("reduceFilterPartials");
    reduceFilterPartials<E><<<gridFor(n), 256, 0, lc.stream>>>(
        ws.partial, n, ws.splits, p.Ci, p.Co, gradLayout(p), static_cast<S *>(filters_grad));
    lc.end();
  }
}

}  // namespace

size_t gatherConvWorkspaceBytes(const ConvProblem &p, GatherDirection dir) {
  return carveGather(p, gatherDims(p, dir), nullptr).bytes;
}

hipError_t launchGatherConv(const LaunchCtx &lc, const ConvProblem &p, GatherDirection dir,
                            const void *gathered, const FilterView &filters, void *workspace,
                            void *result) {
  const GatherDims d = gatherDims(p, dir);
  const GatherWorkspace ws = carveGather(p, d, workspace);
  OffsetCounts inl;
  int max_count = 0;
  hipError_t err = prepareCounts(lc, p, &inl, ws.dev_counts, &max_count);
  if (err != hipSuccess) return err;

  // The MFMA kernel moves rows with 16-byte accesses and packs a partner row
  // into 24 bits of a list entry.
  const bool ptr_ok =
      ((reinterpret_cast<uintptr_t>(gathered) | reinterpret_cast<uintptr_t>(result)) & 15u) == 0;
  const bool use_mfma = mfmaShapeOk(d.Q, d.C) && ptr_ok && d.n_src <= (1 << 24) &&
                        lc.choices.gather_simt != 1;
  switch (p.dtype) {
    case ElemType::kHalf:
      launchGatherTyped<HalfElem>(lc, p, d, ws, inl, max_count, gathered, filters, use_mfma, result);
      break;
    case ElemType::kBFloat16:
      launchGatherTyped<BFloat16Elem>(lc, p, d, ws, inl, max_count, gathered, filters, use_mfma, result);
      break;
    case ElemType::kFloat:
      launchGatherTyped<FloatElem>(lc, p, d, ws, inl, max_count, gathered, filters, use_mfma, result);
      break;
  }
  return hipGetLastError();
}

RowMapShape rowMapShape(const ConvProblem &p, GatherDirection dir) {
  const GatherDims d = gatherDims(p, dir);
  return RowMapShape{p.K, p.L, d.R, d.n_src, d.row_col};
}

// entries [K, rows] | filled-slot counter | per-offset counts [K] (for K beyond the inline limit)
size_t rowMapBytes(int K, int rows) {
  return alignUp((size_t)K * rows * 4) + alignUp(4) + alignUp((size_t)K * 4) + kBaseAlign;
}

hipError_t buildRowMap(const LaunchCtx &lc, const int32_t *indice_pairs, const int64_t *indice_num,
                       const RowMapShape &shape, void *row_map, int32_t *filled_host) {
  const size_t map_elems = (size_t)shape.K * shape.rows;
  int32_t *map = static_cast<int32_t *>(row_map);
  int32_t *counter = reinterpret_cast<int32_t *>(reinterpret_cast<char *>(map) + alignUp(map_elems * 4));
  int32_t *dev_counts = reinterpret_cast<int32_t *>(reinterpret_cast<char *>(counter) + alignUp(4));
  ConvProblem p;
  p.K = shape.K;
  p.L = shape.L;
  p.indice_pairs = indice_pairs;
  p.indice_num = indice_num;
  OffsetCounts inl;
  int max_count = 0;
  hipError_t err = prepareCounts(lc, p, &inl, shape.K > kMaxInlineK ? dev_counts : nullptr, &max_count);
  if (err != hipSuccess) return err;
  lc.begin("fillInt32");
  fillInt32<<<gridFor(map_elems), 256, 0, lc.stream>>>(map, map_elems, -1);
  lc.end();
  fillInt32<<<1, 256, 0, lc.stream>>>(counter, 1, 0);
  if (max_count > 0) {
    lc.begin("scatterRowMap");
    enqueueScatterRowMap(lc, indice_pairs, shape.L, shape.K, inl,
                         shape.K > kMaxInlineK ? dev_counts : nullptr, max_count, shape.row_column,
                         1 - shape.row_column, 0, shape.rows, shape.source_rows, map, nullptr, RunIf{nullptr, 0});
    lc.end();
  }
  if (filled_host == nullptr) return hipGetLastError();
  lc.begin("countFilledSlots");
  countFilledSlots<<<gridFor(map_elems, 1024), 256, 0, lc.stream>>>(map, map_elems, counter);
  lc.end();
  err = hipGetLastError();
  if (err != hipSuccess) return err;
  return hipMemcpyAsync(filled_host, counter, 4, hipMemcpyDeviceToHost, lc.stream);
}

size_t backwardFilterWorkspaceBytes(const ConvProblem &p) {
  return carveFilterGrad(p, nullptr).bytes;
}

bool backwardFilterLaunchesOnly(const ConvProblem &p) { return p.K <= kMaxInlineK; }

hipError_t launchBackwardFilter(const LaunchCtx &lc, const ConvProblem &p, const void *features,
                                const void *output_grad, void *workspace, void *filters_grad) {
  const FilterGradWorkspace ws = carveFilterGrad(p, workspace);
  OffsetCounts inl;
  int max_count = 0;
  hipError_t err = prepareCounts(lc, p, &inl, ws.dev_counts, &max_count);
  if (err != hipSuccess) return err;
  switch (p.dtype) {
    case ElemType::kHalf:
      launchFilterGradTyped<HalfElem>(lc, p, ws, inl, features, output_grad, filters_grad);
      break;
    case ElemType::kBFloat16:
      launchFilterGradTyped<BFloat16Elem>(lc, p, ws, inl, features, output_grad,
                                          filters_grad);
      break;
    case ElemType::kFloat:
      launchFilterGradTyped<FloatElem>(lc, p, ws, inl, features, output_grad, filters_grad);
      break;
  }
  return hipGetLastError();
}

}  // namespace sparse_conv
}  // namespace mluop
