"""Voxels that crowd into one bucket of the grid (coordinates outside it all share one, cells named often do, and those
of a small part of a large grid): the order of a stable sort around the number of voxels that are compared
with each other and around the runs that are sorted beyond it, in a time that stays near that of a spread cloud."""
import numpy as np
import pytest

from test_gpu_order_voxels import BIG

pytestmark = pytest.mark.gpu


def spread(rng, space, voxels):
    lin = np.unique(rng.integers(0, int(np.prod(np.array(space, dtype=np.int64))), 2 * voxels))
    return np.stack(np.unravel_index(rng.permutation(lin)[:voxels], space), axis=1).astype(np.int32)


def crowd(rng, coors, how, count):
    """`count` of the voxels, anywhere in the list, moved together."""
    who = rng.permutation(len(coors))[:count]
    if how == "one cell":
        coors[who] = coors[who[0]]
    elif how == "padding":
        coors[who] = -1
    elif how == "in front":
        coors[who] = rng.integers(-1000, 0, (count, 3))
    elif how == "both ends":
        coors[who] = rng.integers(1 << 20, 1 << 21, (count, 3))
        coors[who[::2]] *= -1
    return coors


def ordered(coors, space):
    import torch
    import mluop_hip
    dev = torch.from_numpy(coors).cuda()
    order, indices = mluop_hip.native().order_voxels(False, dev, list(space), 1)
    torch.cuda.synchronize()
    return order.cpu().numpy(), indices.cpu().numpy()


def check(coors, space):
    c = coors.astype(np.int64)
    want = np.argsort((c[:, 0] * space[1] + c[:, 1]) * space[2] + c[:, 2], kind="stable")
    order, indices = ordered(coors, space)
    assert np.array_equal(order, want)
    assert np.array_equal(indices[:, 1:], coors[want]) and (indices[:, 0] == 1).all()


@pytest.mark.parametrize("how", ["one cell", "padding", "in front", "both ends"])
@pytest.mark.parametrize("voxels,count", [(256, 256), (257, 257), (700, 256), (700, 257), (4095, 4095), (4096, 4096),
                                          (4097, 4097), (20000, 255), (20000, 9001), (40000, 39000)])
def test_crowded_bucket(gpu_handle, how, voxels, count):
    print("crowded bucket", how, voxels, count, flush=True)
    rng = np.random.default_rng(voxels + count)
    check(crowd(rng, spread(rng, BIG, voxels), how, count), BIG)


@pytest.mark.parametrize("voxels", [5000, 70000])
def test_part_of_a_large_grid(gpu_handle, voxels):
    """Cells near each other in a grid whose buckets hold 2^37 cells and more: all voxels in a few of them."""
    print("large grid", voxels, flush=True)
    space = (1 << 19, 1 << 19, 1 << 19)
    rng = np.random.default_rng(voxels)
    check(np.array([7, 300000, 500], np.int32) + spread(rng, (40, 400, 400), voxels), space)


@pytest.mark.parametrize("how", ["padding", "in front"])
def test_time_of_a_crowded_bucket(gpu_handle, how):
    """A tenth of the voxels outside the grid: 1000 to 2100 us when a bucket's voxels were all compared, 30 to 40 us
    where none is crowded."""
    from mluop_hip import nn as spnn
    rng = np.random.default_rng(5)
    handle = spnn._handle()

    def kernels_us(coors):
        totals = []
        for _ in range(4):
            handle.set_kernel_timing(True)
            try:
                ordered(coors, BIG)
                totals.append(sum(ms for _, ms in handle.kernel_timings()) * 1e3)
            finally:
                handle.set_kernel_timing(False)
        return min(totals)

    even = kernels_us(spread(rng, BIG, 120000))
    crowded = kernels_us(crowd(rng, spread(rng, BIG, 120000), how, 12000))
    print("crowded bucket", how, "%.0f us, %.0f without" % (crowded, even), flush=True)
    assert crowded < 8 * even
