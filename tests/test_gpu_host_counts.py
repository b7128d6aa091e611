"""mluOpExtGetIndicePairsHostCounts and mluOpExtGetVoxelizationHostCount: the numbers of what the
handle built, and NOT_SUPPORTED for everything else it can know of."""
import ctypes

import numpy as np
import pytest

from spconv_cases import random_voxels

pytestmark = pytest.mark.gpu

SPACE = (8, 10, 12)


def counts_of(m, handle, pairs, K):
    """(status, counts)"""
    out = (ctypes.c_int64 * K)(*([-7] * K))
    return m.lib().mluOpExtGetIndicePairsHostCounts(handle.ptr, pairs if isinstance(pairs, int) else pairs.data_ptr(),
                                                    K, out), list(out)


def voxel_count_of(m, handle, voxel_num):
    n = ctypes.c_int32(-7)
    return m.lib().mluOpExtGetVoxelizationHostCount(handle.ptr, voxel_num.data_ptr(), ctypes.byref(n)), n.value


def build(m, handle, seed=0, rows=200, ks=(3, 3, 3), sub_m=True):
    import torch
    idx = torch.from_numpy(random_voxels(np.random.default_rng(seed), 1, SPACE, rows)).cuda()
    return m.get_indice_pairs(handle, idx, 1, SPACE, ks, SPACE, [k // 2 for k in ks], [1, 1, 1], [1, 1, 1], sub_m)


def voxelize(m, handle, n=500, voxels=64):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    points = torch.rand((n, 4), device="cuda", generator=g)
    size = torch.tensor([0.25, 0.25, 0.25], device="cuda")
    extent = torch.tensor([0.0, 0.0, 0.0, 1.0, 1.0, 1.0], device="cuda")
    return m.voxelization(handle, points, size, extent, 5, voxels), (points, size, extent)


@pytest.mark.parametrize("ks,sub_m", [((1, 1, 1), True), ((3, 3, 3), True), ((3, 3, 3), False), ((7, 7, 7), True)])
def test_counts_are_those_in_device_memory(gpu_handle, ks, sub_m):
    import mluop_hip as m
    pairs, _, num, _ = build(m, gpu_handle, ks=ks, sub_m=sub_m)
    status, counts = counts_of(m, gpu_handle, pairs, pairs.shape[0])
    assert status == m.STATUS_SUCCESS and counts == num.cpu().tolist()


def test_what_the_handle_did_not_build_is_not_supported(gpu_handle):
    import torch
    import mluop_hip as m
    pairs, _, num, _ = build(m, gpu_handle)
    other = pairs.clone()
    assert counts_of(m, gpu_handle, other, 27)[0] == m.STATUS_NOT_SUPPORTED       # a tensor from elsewhere
    assert counts_of(m, gpu_handle, pairs, 26)[0] == m.STATUS_NOT_SUPPORTED       # another kernel volume
    assert counts_of(m, gpu_handle, pairs.data_ptr() + 4, 27)[0] == m.STATUS_NOT_SUPPORTED
    fresh = m.make_handle_on_current_stream()
    assert counts_of(m, fresh, pairs, 27)[0] == m.STATUS_NOT_SUPPORTED            # another handle's rulebook
    torch.cuda.synchronize()
    fresh.close()
    assert counts_of(m, gpu_handle, pairs, 27) == (m.STATUS_SUCCESS, num.cpu().tolist())


def test_more_offsets_than_are_kept_are_not_supported(gpu_handle):
    import mluop_hip as m
    pairs, _, num, _ = build(m, gpu_handle, rows=60, ks=(7, 7, 8), sub_m=False)
    assert pairs.shape[0] == 392
    assert counts_of(m, gpu_handle, pairs, 392)[0] == m.STATUS_NOT_SUPPORTED
    # the layers' form copies them then
    idx = random_voxels(np.random.default_rng(1), 1, SPACE, 60)
    import torch
    got = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 1, SPACE, (7, 7, 8), SPACE, [3, 3, 4], [1, 1, 1],
                             [1, 1, 1], False, for_layer=True)
    want = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 1, SPACE, (7, 7, 8), SPACE, [3, 3, 4], [1, 1, 1],
                              [1, 1, 1], False)
    assert got[2] == want[2].cpu().tolist()


def test_the_thirty_third_rulebook_takes_the_place_of_the_first(gpu_handle):
    import mluop_hip as m
    kept = [build(m, gpu_handle, seed=s, rows=50 + s) for s in range(33)]
    assert counts_of(m, gpu_handle, kept[0][0], 27)[0] == m.STATUS_NOT_SUPPORTED
    for pairs, _, num, _ in kept[1:]:
        assert counts_of(m, gpu_handle, pairs, 27) == (m.STATUS_SUCCESS, num.cpu().tolist())


def test_captured_calls_are_not_supported(gpu_handle):
    import torch
    import mluop_hip as m
    idx = torch.from_numpy(random_voxels(np.random.default_rng(3), 1, SPACE, 200)).cuda()
    (_, points) = voxelize(m, gpu_handle)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    handle = m.Handle(queue=stream.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        pairs, _, num, _ = m.get_indice_pairs(handle, idx, 1, SPACE, (3, 3, 3), SPACE, [1, 1, 1], [1, 1, 1], [1, 1, 1],
                                              True)
        voxels = m.voxelization(handle, *points, 5, 64)
    assert counts_of(m, handle, pairs, 27)[0] == m.STATUS_NOT_SUPPORTED
    assert voxel_count_of(m, handle, voxels[3])[0] == m.STATUS_NOT_SUPPORTED
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert counts_of(m, handle, pairs, 27)[0] == m.STATUS_NOT_SUPPORTED
        assert voxel_count_of(m, handle, voxels[3])[0] == m.STATUS_NOT_SUPPORTED
    assert int(num.sum()) >= 200 and int(voxels[3]) == 64
    handle.close()


def overwrite(m, handle, how, memory):
    """An operator of the handle that writes into the middle of `memory` (int32, on the device)."""
    import torch
    P = m.lib()
    at = memory.data_ptr() + memory.numel() // 2 * 4 // 256 * 256
    if how == "scatter":
        n = 32
        feats, coors = torch.randn((n, 4), device="cuda"), torch.randint(0, 4, (n, 3), device="cuda", dtype=torch.int32)
        f, c, one = m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_FLOAT, [n, 4]), m.TensorDescriptor(
            m.LAYOUT_ARRAY, m.DTYPE_INT32, [n, 3]), m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_INT32, [1])
        row = m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_INT32, [n])
        size = ctypes.c_size_t(0)
        m.check(P.mluOpGetDynamicPointToVoxelForwardWorkspaceSize(handle.ptr, f.ptr, c.ptr, ctypes.byref(size)))
        ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
        vf, vc, p2v, cnt, num = (torch.empty(s, dtype=torch.int32, device="cuda") for s in ((n, 4), (n, 3), n, n, 1))
        m.check(P.mluOpDynamicPointToVoxelForward(handle.ptr, m.REDUCE_DMEAN, f.ptr, feats.data_ptr(), c.ptr,
                                                  coors.data_ptr(), ws.data_ptr(), size.value, f.ptr, at, c.ptr,
                                                  vc.data_ptr(), row.ptr, p2v.data_ptr(), row.ptr, cnt.data_ptr(),
                                                  one.ptr, num.data_ptr()))
    elif how == "scatter gradient":
        n = 32
        feats, coors = torch.randn((n, 4), device="cuda"), torch.randint(0, 4, (n, 3), device="cuda", dtype=torch.int32)
        vf, vc, p2v, cnt, num = m.dynamic_point_to_voxel_forward(handle, feats, coors, "max")
        f, row = m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_FLOAT, [n, 4]), m.TensorDescriptor(
            m.LAYOUT_ARRAY, m.DTYPE_INT32, [n])
        one = m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_INT32, [1])
        size = ctypes.c_size_t(0)
        m.check(P.mluOpGetDynamicPointToVoxelBackwardWorkspaceSize(handle.ptr, m.REDUCE_DMAX, f.ptr, f.ptr, f.ptr, row.ptr,
                                                                   row.ptr, one.ptr, ctypes.byref(size)))
        ws = torch.empty(size.value + 1, dtype=torch.uint8, device="cuda")
        grad = torch.randn((n, 4), device="cuda")
        m.check(P.mluOpDynamicPointToVoxelBackward(handle.ptr, m.REDUCE_DMAX, f.ptr, grad.data_ptr(), f.ptr,
                                                   feats.data_ptr(), f.ptr, vf.data_ptr(), row.ptr, p2v.data_ptr(), row.ptr,
                                                   cnt.data_ptr(), one.ptr, num.data_ptr(), ws.data_ptr(), size.value,
                                                   f.ptr, at))
    elif how == "voxelization":
        n, v = 100, 16
        points = torch.rand((n, 4), device="cuda")
        vs, cr = torch.full((3,), 0.25, device="cuda"), torch.tensor([0.0, 0, 0, 1, 1, 1], device="cuda")
        D = lambda dtype, dims: m.TensorDescriptor(m.LAYOUT_ARRAY, dtype, dims)  # noqa: E731
        dp, dvs, dcr = D(m.DTYPE_FLOAT, [n, 4]), D(m.DTYPE_FLOAT, [3]), D(m.DTYPE_FLOAT, [6])
        dv, dc, dn, done = (D(m.DTYPE_FLOAT, [v, 2, 4]), D(m.DTYPE_INT32, [v, 3]), D(m.DTYPE_INT32, [v]),
                            D(m.DTYPE_INT32, [1]))
        size = ctypes.c_size_t(0)
        m.check(P.mluOpGetVoxelizationWorkspaceSize(handle.ptr, dp.ptr, dvs.ptr, dcr.ptr, 2, v, 3, True, dv.ptr, dc.ptr,
                                                    dn.ptr, done.ptr, ctypes.byref(size)))
        ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
        c, npv, num = (torch.empty(s, dtype=torch.int32, device="cuda") for s in ((v, 3), v, 1))
        m.check(P.mluOpVoxelization(handle.ptr, dp.ptr, points.data_ptr(), dvs.ptr, vs.data_ptr(), dcr.ptr, cr.data_ptr(),
                                    2, v, 3, True, ws.data_ptr(), size.value, dv.ptr, at, dc.ptr, c.data_ptr(), dn.ptr,
                                    npv.data_ptr(), done.ptr, num.data_ptr()))
    elif how == "row map":
        pairs, _, num, n_out = build(m, handle, seed=9, rows=20)
        d = m.TensorDescriptor(m.LAYOUT_ARRAY, m.DTYPE_INT32, [27, 2, 20])
        size, lost = ctypes.c_size_t(0), ctypes.c_int64(0)
        m.check(P.mluOpExtGetRowMapSize(d.ptr, 20, ctypes.byref(size)))
        assert size.value <= memory.numel() * 2 - 256
        m.check(P.mluOpExtBuildRowMap(handle.ptr, d.ptr, pairs.data_ptr(), (ctypes.c_int64 * 27)(*num.cpu().tolist()), 20,
                                      20, 1, at, size.value, ctypes.byref(lost)))
        m.check(P.mluOpExtForgetRowMap(handle.ptr, at))
    torch.cuda.synchronize()


@pytest.mark.parametrize("how", ["scatter", "scatter gradient", "voxelization", "row map"])
def test_a_rulebook_that_the_handle_wrote_over_is_forgotten(gpu_handle, how):
    """Every operator of the handle, wherever in the pair tensor it writes."""
    import mluop_hip as m
    pairs, _, num, _ = build(m, gpu_handle, rows=400)
    assert counts_of(m, gpu_handle, pairs, 27) == (m.STATUS_SUCCESS, num.cpu().tolist())
    overwrite(m, gpu_handle, how, pairs)
    assert counts_of(m, gpu_handle, pairs, 27)[0] == m.STATUS_NOT_SUPPORTED


def test_voxel_count_is_that_of_the_last_call(gpu_handle):
    import mluop_hip as m
    (first, _), (second, _) = voxelize(m, gpu_handle, 300), voxelize(m, gpu_handle, 12)
    assert voxel_count_of(m, gpu_handle, first[3])[0] == m.STATUS_NOT_SUPPORTED
    assert voxel_count_of(m, gpu_handle, second[3]) == (m.STATUS_SUCCESS, int(second[3]))
    assert voxel_count_of(m, gpu_handle, second[2])[0] == m.STATUS_NOT_SUPPORTED


def test_a_voxel_count_that_the_handle_wrote_over_is_forgotten(gpu_handle):
    import torch
    import mluop_hip as m
    memory = torch.zeros(4096, dtype=torch.int32, device="cuda")
    at = memory[2048:2049]   # where `overwrite` writes
    points = torch.rand((100, 4), device="cuda")
    vs, cr = torch.full((3,), 0.25, device="cuda"), torch.tensor([0.0, 0, 0, 1, 1, 1], device="cuda")
    D = lambda dtype, dims: m.TensorDescriptor(m.LAYOUT_ARRAY, dtype, dims)  # noqa: E731
    dp, dvs, dcr = D(m.DTYPE_FLOAT, [100, 4]), D(m.DTYPE_FLOAT, [3]), D(m.DTYPE_FLOAT, [6])
    dv, dc, dn, done = D(m.DTYPE_FLOAT, [16, 2, 4]), D(m.DTYPE_INT32, [16, 3]), D(m.DTYPE_INT32, [16]), D(m.DTYPE_INT32, [1])
    size = ctypes.c_size_t(0)
    m.check(m.lib().mluOpGetVoxelizationWorkspaceSize(gpu_handle.ptr, dp.ptr, dvs.ptr, dcr.ptr, 2, 16, 3, True, dv.ptr,
                                                      dc.ptr, dn.ptr, done.ptr, ctypes.byref(size)))
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    v, c, npv = (torch.empty(s, dtype=torch.int32, device="cuda") for s in ((16, 2, 4), (16, 3), 16))
    m.check(m.lib().mluOpVoxelization(gpu_handle.ptr, dp.ptr, points.data_ptr(), dvs.ptr, vs.data_ptr(), dcr.ptr,
                                      cr.data_ptr(), 2, 16, 3, True, ws.data_ptr(), size.value, dv.ptr, v.data_ptr(),
                                      dc.ptr, c.data_ptr(), dn.ptr, npv.data_ptr(), done.ptr, at.data_ptr()))
    assert voxel_count_of(m, gpu_handle, at) == (m.STATUS_SUCCESS, int(at))
    overwrite(m, gpu_handle, "scatter", memory)
    assert voxel_count_of(m, gpu_handle, at)[0] == m.STATUS_NOT_SUPPORTED
