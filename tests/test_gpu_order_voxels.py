"""Voxels in the order of their cells: the library's kernels against numpy's stable sort of the cell indices, for
buckets with one voxel, many and all of them, cells outside the grid and cells named twice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = (41, 1504, 1504)


@pytest.mark.parametrize("space,voxels,how", [
    ((1, 1, 2), 2, "grid"), ((4, 16, 16), 1024, "grid"), ((3, 5, 7), 64, "twice"), ((5, 33, 31), 5115, "grid"),
    (BIG, 2, "grid"), (BIG, 255, "grid"), (BIG, 257, "cluster"), (BIG, 43000, "grid"), (BIG, 43000, "cluster"),
    (BIG, 5000, "outside"), (BIG, 3000, "one"), ((2, 3, 4), 3000, "outside"), (BIG, 262145, "grid"),
    (BIG, 1 << 20, "grid"), ((1 << 19, 1 << 19, 1 << 19), 4000, "grid")])
def test_order_of_a_stable_sort(gpu_handle, space, voxels, how):
    import torch
    from mluop_hip import nn as spnn
    print("order voxels", space, voxels, how, flush=True)
    rng = np.random.default_rng(voxels)
    cells = int(np.prod(np.array(space, dtype=object)))
    if how == "grid":
        lin = rng.permutation(cells)[:voxels] if cells < 1 << 22 else rng.permutation(np.unique(rng.integers(0, cells, voxels)))
    elif how == "cluster":  # runs along a few rows of the grid
        lin = rng.permutation(np.unique((rng.integers(0, 40, voxels) * 977 * 1504 + rng.integers(0, 1500, voxels))))
    else:
        lin = rng.integers(0, cells, voxels)
    coors = np.stack(np.unravel_index(lin, space), axis=1).astype(np.int32)
    if how == "outside":
        coors = rng.integers(-(1 << 31), 1 << 31, coors.shape).astype(np.int32)
        coors[::3] %= np.array(space, np.int32)
    elif how == "one":
        coors[:] = coors[0]
    c = coors.astype(np.int64)
    with np.errstate(over="ignore"):
        order = np.argsort((c[:, 0] * space[1] + c[:, 1]) * space[2] + c[:, 2], kind="stable")
    feats = torch.arange(len(coors) * 3, device="cuda", dtype=torch.float32).view(-1, 3).requires_grad_(True)
    dev = torch.from_numpy(coors).cuda()
    assert spnn._ordered_by_library(dev, space, 3)
    t = spnn.sparse_tensor_from_voxels(feats, dev, space, batch_index=3, batch_size=4)
    torch.cuda.synchronize()
    assert t.indices.dtype == torch.int32 and (t.indices[:, 0] == 3).all()
    assert (t.indices[:, 1:].cpu().numpy() == coors[order]).all()
    assert (t.features.detach()[:, 0].cpu().numpy().astype(np.int64) == order * 3).all()
    scale = torch.arange(len(coors), device="cuda", dtype=torch.float32).view(-1, 1)
    (t.features * scale).sum().backward()
    place = np.empty_like(order)
    place[order] = np.arange(len(order))
    assert (feats.grad[:, 2].cpu().numpy() == place).all()
