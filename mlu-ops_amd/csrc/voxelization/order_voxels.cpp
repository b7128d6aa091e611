// mluOpExtOrderVoxels and its workspace query (no counterpart in the reference).
#include "core/core.h"
#include "mlu_op_ext.h"
#include "voxelization/order_voxels.h"

namespace {

mluOpStatus_t shapeOf(const char *api, int64_t voxels, const int64_t space[3], int32_t batch_index,
                      mluop::voxelization::OrderShape *s) {
  PARAM_CHECK(api, voxels > 0);
  PARAM_CHECK(api, space != NULL);
  int64_t cells = 1;
  for (int a = 0; a < 3; ++a) {
    PARAM_CHECK(api, space[a] > 0 && space[a] <= INT32_MAX);
    PARAM_CHECK(api, cells <= ((int64_t)1 << 62) / space[a]);
    cells *= space[a];
    s->space[a] = space[a];
  }
  if (voxels > mluop::voxelization::kMaxOrderedVoxels) {
    MLUOP_LOG(ERROR) << api << " At most " << mluop::voxelization::kMaxOrderedVoxels
                     << " voxels per call are supported.";
    return MLUOP_STATUS_NOT_SUPPORTED;
  }
  s->voxels = voxels;
  s->batch_index = batch_index;
  return MLUOP_STATUS_SUCCESS;
}

}  // namespace

mluOpStatus_t MLUOP_WIN_API mluOpExtGetOrderVoxelsWorkspaceSize(int64_t voxels, const int64_t space[3],
                                                                size_t *size) {
  const char *api = "[mluOpExtGetOrderVoxelsWorkspaceSize]";
  PARAM_CHECK(api, size != NULL);
  mluop::voxelization::OrderShape s;
  const mluOpStatus_t status = shapeOf(api, voxels, space, 0, &s);
  if (status != MLUOP_STATUS_SUCCESS) return status;
  *size = mluop::voxelization::orderVoxelsWorkspaceBytes(s);
  return MLUOP_STATUS_SUCCESS;
}

mluOpStatus_t MLUOP_WIN_API mluOpExtOrderVoxels(mluOpHandle_t handle, const void *coors, int64_t voxels,
                                                const int64_t space[3], int32_t batch_index, void *workspace,
                                                size_t workspace_size, void *order, void *indices) {
  const char *api = "[mluOpExtOrderVoxels]";
  PARAM_CHECK(api, handle != NULL);
  mluop::voxelization::OrderShape s;
  const mluOpStatus_t status = shapeOf(api, voxels, space, batch_index, &s);
  if (status != MLUOP_STATUS_SUCCESS) return status;
  PARAM_CHECK(api, coors != NULL);
  PARAM_CHECK(api, workspace != NULL);
  PARAM_CHECK(api, order != NULL);
  PARAM_CHECK(api, indices != NULL);
  PARAM_CHECK(api, workspace_size >= mluop::voxelization::orderVoxelsWorkspaceBytes(s));
  DEVICE_HANDLE_CHECK(api, handle);
  HIP_CHECK_RETURN(api, hipSetDevice(handle->device));
  handle->forgetNotesIn(order, (size_t)voxels * sizeof(int64_t));
  handle->forgetNotesIn(indices, (size_t)voxels * 4 * sizeof(int32_t));
  handle->forgetNotesIn(workspace, workspace_size);
  HIP_CHECK_RETURN(api, mluop::voxelization::launchOrderVoxels(
                            handle->launchCtx(), s, static_cast<const int32_t *>(coors), workspace,
                            static_cast<int64_t *>(order), static_cast<int32_t *>(indices)));
  return MLUOP_STATUS_SUCCESS;
}
