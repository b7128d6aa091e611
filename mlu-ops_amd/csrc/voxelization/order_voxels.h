// Host-side interface of the kernels that order voxels by their cell of the grid.
#ifndef MLUOP_AMD_VOXELIZATION_ORDER_VOXELS_H_
#define MLUOP_AMD_VOXELIZATION_ORDER_VOXELS_H_

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "core/launch.h"

namespace mluop {
namespace voxelization {

// Most voxels one call accepts: a voxel of a crowded bucket is looked up in all its runs of 4096, and
// coordinates outside the grid all share a bucket.
constexpr int64_t kMaxOrderedVoxels = (int64_t)1 << 20;

struct OrderShape {
  int64_t voxels;    // [1, kMaxOrderedVoxels]
  int64_t space[3];  // cells along (z, y, x), their product below 2^62
  int32_t batch_index;
};

size_t orderVoxelsWorkspaceBytes(const OrderShape &s);

hipError_t launchOrderVoxels(const LaunchCtx &lc, const OrderShape &s, const int32_t *coors, void *workspace,
                             int64_t *order, int32_t *indices);

}  // namespace voxelization
}  // namespace mluop

#endif  // MLUOP_AMD_VOXELIZATION_ORDER_VOXELS_H_
