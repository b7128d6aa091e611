// Host-side interface of the hard-voxelization kernel set.
#ifndef MLUOP_AMD_VOXELIZATION_VOXELIZE_H_
#define MLUOP_AMD_VOXELIZATION_VOXELIZE_H_

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "core/launch.h"

namespace mluop {
namespace voxelization {

struct VoxelizeShape {
  int64_t num_points;
  int num_features;
  int max_points;
  int max_voxels;
};

// Most points one call accepts (a bucket's table has up to three slots a point,
// counted in 32 bits).
constexpr int64_t kMaxPoints = (int64_t)1 << 28;

// Bytes of device workspace: the per-point arrays and the cell tables.
size_t voxelizeWorkspaceBytes(const VoxelizeShape &s);

// Enqueues the whole operator: outputs zero-filled, then written.  The number of voxels also goes,
// below the low half of `stamp`, into `host_voxel_num` (pinned host memory; null: nowhere).
hipError_t launchVoxelize(const LaunchCtx &lc, const VoxelizeShape &s, const float *points,
                          const float *voxel_size, const float *coors_range, void *workspace,
                          size_t workspace_bytes, float *voxels, int32_t *coors,
                          int32_t *num_points_per_voxel, int32_t *voxel_num, unsigned long long *host_voxel_num,
                          unsigned long long stamp);

}  // namespace voxelization
}  // namespace mluop

#endif  // MLUOP_AMD_VOXELIZATION_VOXELIZE_H_
