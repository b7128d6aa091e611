// Host-side interface of the rulebook (indice pairs) kernel set.
#ifndef MLUOP_AMD_SPARSE_CONV_RULEBOOK_H_
#define MLUOP_AMD_SPARSE_CONV_RULEBOOK_H_

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "core/launch.h"

namespace mluop {
namespace sparse_conv {

// Geometry of one sparse convolution, axes in (d, h, w) order.
struct RulebookGeom {
  int batch;
  int in_space[3];
  int out_space[3];
  int ksize[3];
  int pad[3];
  int stride[3];
  int dilation[3];
  int K;         // kernel volume
  int L;         // active input rows
  int out_rows;  // rows of the caller's out_indices tensor (M)
  bool sub_m;
  // Pair slots behind an offset's pairs become -1, as the operator promises; a caller who reads no
  // further than indice_num leaves them as they are (at 125 offsets of 400 000 rows, 403 of the 453 MB that
  // the probe writes).
  bool fill_tails = true;
};

// Where the last kernel of a rulebook reports (pinned host memory, written from the device), in
// words that carry the low half of the stamp above their value, so that a reader sees by
// itself whether a word is this rulebook's.  Null pointers: no report.
struct RulebookReportTarget {
  // were the input rows strictly ascending in (n, d, h, w) order?
  unsigned long long *order_word = nullptr;
  // A value no earlier rulebook of any handle used (never 0); also marks this call's words
  // in the workspace, so it is set whether or not a report is wanted.
  unsigned long long stamp = 0;
  // word k: the number of pairs of offset k
  unsigned long long *count_words = nullptr;
};

// A value with the low half of a stamp above it, as the device stores it for the host.
#if defined(__HIPCC__)
__host__ __device__
#endif
inline unsigned long long stampedWord(unsigned long long stamp, int value) {
  return (stamp << 32) | (unsigned int)value;
}

// Bytes of device workspace the kernel set needs for this geometry.
size_t rulebookWorkspaceBytes(const RulebookGeom &g);

// Enqueues submanifold rulebook construction on the context's stream.
hipError_t launchSubmRulebook(const LaunchCtx &lc, const RulebookGeom &g, const int32_t *indices,
                              void *workspace, int32_t *indice_pairs, int32_t *out_indices,
                              int32_t *indice_num, const RulebookReportTarget &report);

// Enqueues regular (strided / dilated) rulebook construction.  The kernel that numbers the
// output cells stores their count, stamped, into `host_num_act_out` (pinned host memory): the
// caller waits for that word, while the kernel that writes the pair lists may still be
// running.
hipError_t launchRegularRulebook(const LaunchCtx &lc, const RulebookGeom &g,
                                 const int32_t *indices, void *workspace, int32_t *indice_pairs,
                                 int32_t *out_indices, int32_t *indice_num,
                                 unsigned long long *host_num_act_out,
                                 const RulebookReportTarget &report);

}  // namespace sparse_conv
}  // namespace mluop

#endif  // MLUOP_AMD_SPARSE_CONV_RULEBOOK_H_
