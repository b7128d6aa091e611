// Host-side interface of the dynamic point-to-voxel (forward) kernel set.
#ifndef MLUOP_AMD_DYNAMIC_POINT_TO_VOXEL_SCATTER_POINTS_H_
#define MLUOP_AMD_DYNAMIC_POINT_TO_VOXEL_SCATTER_POINTS_H_

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "core/launch.h"

namespace mluop {
namespace dynamic_point_to_voxel {

struct ScatterShape {
  int num_points;    // N
  int num_features;  // C
  int voxel_rows;    // rows of the voxel_* output tensors (<= N)
  bool reduce_max;   // max, else mean
};

size_t scatterWorkspaceBytes(const ScatterShape &s);

// Enqueues the operator.  It waits once for the largest coordinate of every axis, which the first
// kernels store below the low half of `stamp` into `host_words` (three words of pinned host
// memory) and which sizes the radix sorts.
hipError_t launchScatterPoints(const LaunchCtx &lc, const ScatterShape &s, const float *feats,
                               int32_t *coors, void *workspace, size_t workspace_bytes,
                               unsigned long long *host_words, unsigned long long stamp, float *voxel_feats,
                               int32_t *voxel_coors, int32_t *point2voxel_map, int32_t *voxel_points_count,
                               int32_t *voxel_num);

// Backward of the max reduction: `workspace` holds voxel_rows * num_features ints at least.
hipError_t launchScatterPointsBackward(const LaunchCtx &lc, int num_points, int num_features,
                                       int voxel_rows, const float *grad_voxel_feats,
                                       const float *feats, const float *voxel_feats,
                                       const int32_t *point2voxel_map, const int32_t *voxel_num,
                                       void *workspace, size_t workspace_bytes, float *grad_feats);

}  // namespace dynamic_point_to_voxel
}  // namespace mluop

#endif  // MLUOP_AMD_DYNAMIC_POINT_TO_VOXEL_SCATTER_POINTS_H_
