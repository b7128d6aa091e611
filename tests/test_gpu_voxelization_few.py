"""Clouds of few points, which the voxelizer takes in three launches: edges of their rounds and of their range, buckets
beyond the list and the table in LDS, on either side of the range.  Bit for bit against the sort-based formulation
that the CPU tests pin to the oracle."""
import numpy as np
import pytest

from test_gpu_voxelization import assert_same, run_gpu
from test_gpu_voxelization_partition import COARSE, FINE, bucket_of
from voxel_cases import lidar_like_points, sorted_voxelization

pytestmark = pytest.mark.gpu

FEW = 1 << 16


@pytest.mark.parametrize("n", [1, 16, 17, 8191, 8192, 8193, 16385, 24577, FEW - 1, FEW, FEW + 1])
@pytest.mark.parametrize("grid", ["coarse", "fine"])
def test_edges_of_rounds_and_range(gpu_handle, n, grid):
    vs, cr = COARSE if grid == "coarse" else FINE
    rng = np.random.default_rng(n)
    pts = lidar_like_points(rng, n, features=4, spread=(8.0, 4.0, 2.0))
    pts[n // 2:, :3] = pts[:n - n // 2, :3]     # every cell of the first half again
    print("voxelization", n, grid, flush=True)
    assert_same(run_gpu(gpu_handle, pts, vs, cr, 3, 40000), sorted_voxelization(pts, vs, cr, 3, 40000))


def tag_of(key):
    """The bucket a cell of a small cloud is in."""
    return (bucket_of(key, 1 << 32).astype(np.uint64) * np.uint64(255)) >> np.uint64(32)


@pytest.mark.parametrize("cells", [510, 512, 514, 1024, 1026, 1536, 2048, 5000])
@pytest.mark.parametrize("few", [True, False])
def test_buckets_with_more_cells_than_lds_holds(gpu_handle, cells, few):
    """Cells of one bucket, twice each: around the 1024 points of the list and what the table in LDS takes.  Points outside
    the grid make up a cloud beyond the range, whose 128 buckets are others."""
    rng = np.random.default_rng(cells)
    side = 128
    keys = np.arange(side ** 3)
    keys = rng.permutation(keys[(tag_of(keys) == 5) if few else (bucket_of(keys, 128) == 5)])[:cells]
    assert len(keys) == cells
    keys = np.concatenate([keys, keys])
    rng.shuffle(keys)
    pts = np.stack([keys % side, keys // side % side, keys // side ** 2, keys], 1).astype(np.float32)
    pts[:, :3] += 0.5
    if not few:
        outside = np.full((70000 - len(pts), 4), -5.0, np.float32)
        pts = rng.permutation(np.concatenate([pts, outside]))
    vs, cr = [1.0, 1.0, 1.0], [0.0, 0.0, 0.0, float(side), float(side), float(side)]
    for max_points in (1, 3):
        assert_same(run_gpu(gpu_handle, pts, vs, cr, max_points, 6000), sorted_voxelization(pts, vs, cr, max_points, 6000))


@pytest.mark.parametrize("max_points", [1, 20, 700])
@pytest.mark.parametrize("grid", ["coarse", "fine"])
def test_crowded_cells_beyond_the_range(gpu_handle, max_points, grid):
    vs, cr = COARSE if grid == "coarse" else FINE
    rng = np.random.default_rng(max_points)
    pts = lidar_like_points(rng, FEW + 5000, features=4, spread=(8.0, 4.0, 2.0))
    crowded = rng.random(len(pts))
    pts[crowded < 0.1, :3] = (1.1, 0.1, 0.1)
    pts[crowded > 0.9, :3] = (5.1, 0.1, 0.1)
    for n in (FEW - 3000, len(pts)):
        assert_same(run_gpu(gpu_handle, pts[:n], vs, cr, max_points, 40000),
                    sorted_voxelization(pts[:n], vs, cr, max_points, 40000))


@pytest.mark.parametrize("cells", [1, 32, 33, 510, 512, 514, 1026, 3000])
def test_buckets_of_grids_with_64_bit_keys(gpu_handle, cells):
    """Cells of one bucket, twice each, in a grid of 2^33 cells: the table in LDS has 64-bit keys there, and those of whole
    rounds differ in their upper halves only."""
    rng = np.random.default_rng(cells)
    side = 2048
    keys = np.unique(rng.integers(0, side ** 3, 400 * cells + 2000))
    keys = np.concatenate([keys, keys[keys < 1 << 32] + (1 << 32)])
    keys = rng.permutation(np.unique(keys[tag_of(keys) == 5]))[:cells]
    assert len(keys) == cells and keys.max() < side ** 3
    keys = np.concatenate([keys, keys])
    rng.shuffle(keys)
    pts = np.stack([keys % side, keys // side % side, keys // side ** 2, keys], 1).astype(np.float32)
    pts[:, :3] += 0.5
    vs, cr = [1.0, 1.0, 1.0], [0.0, 0.0, 0.0, float(side), float(side), float(side)]
    print("voxelization, long keys", cells, flush=True)
    for max_points in (1, 3):
        assert_same(run_gpu(gpu_handle, pts, vs, cr, max_points, 6000), sorted_voxelization(pts, vs, cr, max_points, 6000))
