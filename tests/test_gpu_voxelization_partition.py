"""The partition of the voxelizer at its edges: tiles, rounds of a tile, buckets beyond the table in LDS,
grids whose cell numbers need 64 bits.  Bit for bit against the CPU oracle, large clouds against the
sort-based formulation that the CPU tests pin to it."""
import numpy as np
import pytest

import voxelization_oracle as vox
from test_gpu_voxelization import assert_same, run_gpu
from voxel_cases import lidar_like_points, sorted_voxelization

pytestmark = pytest.mark.gpu

COARSE = ([0.4, 0.4, 1.0], [0.0, -4.0, -2.0, 8.0, 4.0, 1.0])
FINE = ([0.0005, 0.0005, 0.0005], [0.0, -4.0, -2.0, 8.0, 4.0, 1.0])   # 1.5e12 cells


@pytest.mark.parametrize("n", [1, 63, 65, 511, 513, 2047, 2049, 4097, 12289])
@pytest.mark.parametrize("grid", ["coarse", "fine"])
def test_edges_of_tiles(gpu_handle, n, grid):
    vs, cr = COARSE if grid == "coarse" else FINE
    rng = np.random.default_rng(n)
    pts = lidar_like_points(rng, n, features=5, spread=(8.0, 4.0, 2.0))
    pts[n // 2:, :3] = pts[:n - n // 2, :3]     # every cell of the first half again
    print("voxelization", n, grid, flush=True)
    assert_same(run_gpu(gpu_handle, pts, vs, cr, 3, 5000), vox.voxelization(pts, vs, cr, 3, 5000))


@pytest.mark.parametrize("max_points", [1, 20, 700])
@pytest.mark.parametrize("grid", ["coarse", "fine"])
def test_buckets_with_more_points_than_the_table_in_lds(gpu_handle, max_points, grid):
    vs, cr = COARSE if grid == "coarse" else FINE
    rng = np.random.default_rng(max_points)
    pts = lidar_like_points(rng, 9000, features=4, spread=(8.0, 4.0, 2.0))
    crowded = rng.random(9000)
    pts[crowded < 0.3, :3] = (1.1, 0.1, 0.1)    # padding at one place
    pts[crowded > 0.8, :3] = (5.1, 0.1, 0.1)
    assert_same(run_gpu(gpu_handle, pts, vs, cr, max_points, 4000), vox.voxelization(pts, vs, cr, max_points, 4000))


@pytest.mark.parametrize("n", [2_100_001, 4_300_000, 6_100_000])
def test_several_rounds_a_tile_and_scanned_tiles(gpu_handle, n):
    rng = np.random.default_rng(5)
    pts = lidar_like_points(rng, n, features=3, spread=(70.4, 40.0, 3.0), outliers=0.05)
    vs, cr = [0.05, 0.05, 0.1], [0.0, -40.0, -3.0, 70.4, 40.0, 1.0]
    assert_same(run_gpu(gpu_handle, pts, vs, cr, 5, 150000), sorted_voxelization(pts, vs, cr, 5, 150000))


def bucket_of(key, buckets):
    """The bucket a cell is hashed to."""
    k = key.astype(np.uint64)
    k ^= k >> np.uint64(33)
    k *= np.uint64(0xff51afd7ed558ccd)
    k ^= k >> np.uint64(33)
    k *= np.uint64(0xc4ceb9fe1a85ec53)
    k ^= k >> np.uint64(33)
    return (k & np.uint64(buckets - 1)).astype(np.int64)


@pytest.mark.parametrize("cells", [1023, 1025, 1535, 1536, 1537, 1600, 2048, 5000])
def test_buckets_with_more_cells_than_the_table_in_lds(gpu_handle, cells):
    """A cloud whose cells fall into one of its 64 buckets, around the number that the table in LDS takes
    (2048 slots, 512 of them left over), every cell with one point or two."""
    rng = np.random.default_rng(cells)
    side = 128
    keys = np.arange(side ** 3)
    keys = rng.permutation(keys[bucket_of(keys, 64) == 5])[:cells]
    keys = np.concatenate([keys, keys[:cells // 3]])
    rng.shuffle(keys)
    pts = np.stack([keys % side, keys // side % side, keys // side ** 2, keys], 1).astype(np.float32)
    pts[:, :3] += 0.5
    vs, cr = [1.0, 1.0, 1.0], [0.0, 0.0, 0.0, float(side), float(side), float(side)]
    for max_points in (1, 3):
        assert_same(run_gpu(gpu_handle, pts, vs, cr, max_points, 6000), sorted_voxelization(pts, vs, cr, max_points, 6000))
