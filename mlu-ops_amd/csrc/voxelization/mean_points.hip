// mluOpExtMeanVoxelPoints (no counterpart in the reference): the mean of every voxel's points in one launch.
#include <hip/hip_runtime.h>

#include "core/core.h"
#include "mlu_op_ext.h"

namespace {

constexpr int kThreads = 256;

// V consecutive features of a voxel per thread: the sum of all its slots (those behind its points are zeros, as the
// voxelizer leaves them) in four running sums, over the number of its points or one.
// Bound by the lines its requests touch (every slot of a voxel is a request of its own over the same lines).  120 000
// voxels of 5 points and 5 features, us of kernels: as a sum, a clamp, a conversion and a division 23.4 in four launches,
// this 8.6 in one; eight slots requested at once, behind the last one clamped, 10.8.
template <int V>
__global__ __launch_bounds__(kThreads) void meanVoxelPoints(const float *__restrict__ voxels,
                                                            const int32_t *__restrict__ counts,
                                                            uint32_t vectors, int max_points,
                                                            uint32_t vectors_per_row,
                                                            float *__restrict__ mean) {
  typedef float Vector __attribute__((ext_vector_type(V)));
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= vectors) return;
  const uint32_t voxel = i / vectors_per_row;
  const Vector *at = reinterpret_cast<const Vector *>(voxels) +
                     ((uint64_t)voxel * ((uint64_t)max_points * vectors_per_row) + (i - voxel * vectors_per_row));
  const int32_t points = counts[voxel];
  Vector sums[4] = {};
  int p = 0;
  for (; p + 4 <= max_points; p += 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sums[j] += at[(uint64_t)(p + j) * vectors_per_row];
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (p + j < max_points) sums[j] += at[(uint64_t)(p + j) * vectors_per_row];
  const Vector sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
  reinterpret_cast<Vector *>(mean)[i] = sum / (float)(points < 1 ? 1 : points);
}

}  // namespace

mluOpStatus_t MLUOP_WIN_API mluOpExtMeanVoxelPoints(mluOpHandle_t handle, const void *voxels,
                                                    const void *num_points_per_voxel, int64_t num_voxels,
                                                    int32_t max_points, int32_t features, void *mean) {
  const char *api = "[mluOpExtMeanVoxelPoints]";
  PARAM_CHECK(api, handle != NULL);
  PARAM_CHECK(api, num_voxels > 0);
  PARAM_CHECK(api, max_points > 0);
  PARAM_CHECK(api, features > 0);
  PARAM_CHECK(api, num_voxels <= INT32_MAX / features);
  PARAM_CHECK(api, voxels != NULL);
  PARAM_CHECK(api, num_points_per_voxel != NULL);
  PARAM_CHECK(api, mean != NULL);
  DEVICE_HANDLE_CHECK(api, handle);
  HIP_CHECK_RETURN(api, hipSetDevice(handle->device));
  handle->forgetNotesIn(mean, (size_t)num_voxels * features * sizeof(float));
  const bool fours = features % 4 == 0 && (reinterpret_cast<uintptr_t>(voxels) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(mean) & 15) == 0;
  const int per_row = fours ? features / 4 : features;
  const uint32_t vectors = (uint32_t)(num_voxels * per_row);
  const unsigned blocks = (vectors + kThreads - 1) / kThreads;
  auto kernel = fours ? meanVoxelPoints<4> : meanVoxelPoints<1>;
  const mluop::LaunchCtx lc = handle->launchCtx();
  lc.begin("meanVoxelPoints");
  kernel<<<blocks, kThreads, 0, lc.stream>>>(static_cast<const float *>(voxels),
                                             static_cast<const int32_t *>(num_points_per_voxel), vectors, max_points,
                                             (uint32_t)per_row, static_cast<float *>(mean));
  lc.end();
  HIP_CHECK_RETURN(api, hipGetLastError());
  return MLUOP_STATUS_SUCCESS;
}
