"""Point scatter with features taken one, two and four at a time by a thread; a backward pass by atomic
minima, and by lists of points with voxels on both sides of the longest list and of the points a
thread holds at once, with and without room for the lists."""
import ctypes

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
    for rows in (n, (n + 1) // 2):   # (half the rows: points of voxels without a row)
        vf, vc, p2v, cnt, num = mluop_hip.dynamic_point_to_voxel_forward(gpu_handle, tf, tc.clone(), "max", rows)
        grad = mluop_hip.dynamic_point_to_voxel_backward(gpu_handle, torch.from_numpy(g[:rows]).cuda(), tf, vf, p2v,
                                                         cnt, num)
        torch.cuda.synchronize()
        want = dpv.backward(g[:rows], feats, vf.cpu().numpy(), p2v.cpu().numpy(), int(num.item()))
        assert np.array_equal(grad.cpu().numpy(), want), rows


def crowded(rng, n, crowds):
    """Coordinates of n points: a voxel of each size in `crowds`, the rest in voxels of a few points."""
    cell = np.repeat(np.arange(len(crowds)), crowds)[:n]
    cell = np.concatenate([cell, rng.integers(1000, 1000 + n, n - cell.size)])
    cell[rng.random(n) < 0.02] = -1
    rng.shuffle(cell)
    return np.where(cell[:, None] < 0, -1, np.stack([cell // 10000, cell // 100 % 100, cell % 100], 1)).astype(np.int32)


def check_backward(gpu_handle, rng, feats, coors):
    import torch
    import mluop_hip
    g = rng.standard_normal(feats.shape).astype(np.float32)
    tf, tc = torch.from_numpy(feats).cuda(), torch.from_numpy(coors).cuda()
    vf, vc, p2v, cnt, num = mluop_hip.dynamic_point_to_voxel_forward(gpu_handle, tf, tc.clone(), "max")
    grad = mluop_hip.dynamic_point_to_voxel_backward(gpu_handle, torch.from_numpy(g).cuda(), tf, vf, p2v, cnt, num)
    torch.cuda.synchronize()
    assert np.array_equal(grad.cpu().numpy(), dpv.backward(g, feats, vf.cpu().numpy(), p2v.cpu().numpy(), int(num.item())))


@pytest.mark.parametrize("c", [3, 32, 65])
@pytest.mark.parametrize("n,crowds", [(33, [33]), (2049, [2049]), (6000, [3000]), (20000, [12000, 33, 32])])
def test_backward_with_crowded_voxels(gpu_handle, c, n, crowds):
    rng = np.random.default_rng(c + n)
    coors = crowded(rng, n, crowds)
    for feats in (rng.standard_normal((n, c)).astype(np.float32), np.zeros((n, c), np.float32)):
        feats[rng.random(n) < 0.01] = np.nan
        check_backward(gpu_handle, rng, feats, coors)


@pytest.mark.parametrize("c,n,crowds", [
    (32, 250_000, [33, 32, 31, 34, 1, 2, 4, 5, 100_000]),     # lists beside one voxel without, and around the limit
    (33, 245_000, [40] * 3000),                               # one feature a thread; most points without a list
    (34, 240_000, [31] * 3000),                               # two; most in long lists
    (64, 125_001, []),                                        # short lists only
    (128, 62_500, [62_500]),                                  # so few voxels that nothing is listed
    (32, 250_000, [250] * 900),
])
def test_backward_of_many_wide_features(gpu_handle, c, n, crowds):
    """Sizes at which the points are listed: voxels on both sides of the longest list."""
    rng = np.random.default_rng(c + n)
    coors = crowded(rng, n, crowds)
    feats = rng.integers(-8, 9, (n, c)).astype(np.float32)   # ties in every longer list
    feats[rng.random(n) < 0.01] = np.nan
    check_backward(gpu_handle, rng, feats, coors)


@pytest.mark.parametrize("rows", [1000, 100_000])
def test_backward_with_no_more_workspace_than_it_must_have(gpu_handle, rows):
    """rows x features words: room for the lists beside many rows, not beside few."""
    import torch
    import mluop_hip as m
    n, c = 250_000, 32
    rng = np.random.default_rng(rows)
    coors = crowded(rng, n, [100, 40, 3])
    feats = rng.integers(-8, 9, (n, c)).astype(np.float32)
    g = torch.from_numpy(rng.standard_normal((rows, c)).astype(np.float32)).cuda()
    tf = torch.from_numpy(feats).cuda()
    vf, vc, p2v, cnt, num = m.dynamic_point_to_voxel_forward(gpu_handle, tf, torch.from_numpy(coors).cuda(), "max", rows)

    def desc(dtype, *dims):
        return m.TensorDescriptor(m.LAYOUT_ARRAY, dtype, dims)
    wide, points, lines, line = (desc(m.DTYPE_FLOAT, rows, c), desc(m.DTYPE_FLOAT, n, c), desc(m.DTYPE_INT32, n),
                                 desc(m.DTYPE_INT32, rows))
    one = desc(m.DTYPE_INT32, 1)
    guard = torch.full((rows * c + 64,), 0x5a5a5a5a, dtype=torch.int32, device="cuda")   # 64 words behind the workspace
    grad = torch.empty((n, c), device="cuda")
    gpu_handle.set_kernel_timing(True)
    m.check(m.lib().mluOpDynamicPointToVoxelBackward(
        gpu_handle.ptr, m.REDUCE_DMAX, wide.ptr, g.data_ptr(), points.ptr, tf.data_ptr(), wide.ptr, vf.data_ptr(), lines.ptr,
        p2v.data_ptr(), line.ptr, cnt.data_ptr(), one.ptr, num.data_ptr(), ctypes.c_void_p(guard.data_ptr()), rows * c * 4,
        points.ptr, grad.data_ptr()))
    listed = any(k == "dpvBackwardLists" for k, _ in gpu_handle.kernel_timings())
    gpu_handle.set_kernel_timing(False)
    torch.cuda.synchronize()
    assert listed == (rows == 100_000)
    assert bool((guard[rows * c:] == 0x5a5a5a5a).all())
    want = dpv.backward(g.cpu().numpy(), feats, vf.cpu().numpy(), p2v.cpu().numpy(), min(int(num.item()), rows))
    assert np.array_equal(grad.cpu().numpy(), want)
