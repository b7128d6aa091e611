"""Point scatter with features taken one, two and four at a time by a thread, voxels on both sides of
the points a thread holds at once, and a backward pass with and without room for the point lists."""
import numpy as np
import pytest

import dynamic_point_to_voxel_oracle as dpv
from test_gpu_dynamic_point_to_voxel import assert_same, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [1, 2, 3, 4, 6, 9, 32])
@pytest.mark.parametrize("n,span", [(1, 1), (700, 3), (3001, 8), (9000, 40)])
def test_forward_and_backward(gpu_handle, c, n, span):
    import torch
    import mluop_hip
    rng = np.random.default_rng(c * n)
    feats = rng.integers(-3, 4, (n, c)).astype(np.float32)   # ties everywhere
    coors = rng.integers(0, span, (n, 3)).astype(np.int32)
    coors[rng.random(n) < 0.1] = -1
    for mode in ("max", "mean"):
        assert_same(run_gpu(gpu_handle, mode, feats, coors), dpv.forward(mode, feats, coors))
    g = rng.standard_normal((n, c)).astype(np.float32)
    tf, tc = torch.from_numpy(feats).cuda(), torch.from_numpy(coors).cuda()
    for rows in (n, (n + 1) // 2):   # (half the rows: less workspace, and points of voxels without a row)
        vf, vc, p2v, cnt, num = mluop_hip.dynamic_point_to_voxel_forward(gpu_handle, tf, tc.clone(), "max", rows)
        grad = mluop_hip.dynamic_point_to_voxel_backward(gpu_handle, torch.from_numpy(g[:rows]).cuda(), tf, vf, p2v,
                                                         cnt, num)
        torch.cuda.synchronize()
        want = dpv.backward(g[:rows], feats, vf.cpu().numpy(), p2v.cpu().numpy(), int(num.item()))
        assert np.array_equal(grad.cpu().numpy(), want), rows
