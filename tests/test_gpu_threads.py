"""Layers used by several threads on one stream.  All of them go through the one library handle of that
stream: what a call leaves there for its host (stamps, the row count of a strided rulebook, pair
counts, the number of voxels, row maps and settings) must not meet another thread's."""
import threading

import numpy as np
import pytest

from spconv_cases import random_voxels

pytestmark = pytest.mark.gpu

SPACE = (12, 20, 24)


def make_job(seed):
    """One program with a cloud of its own: strided, submanifold and inverse layer, and a voxelizer."""
    import torch
    from mluop_hip import nn as spnn
    rng = np.random.default_rng(seed)
    rows = 300 + 150 * seed
    idx = torch.from_numpy(random_voxels(rng, 1, SPACE, rows)).cuda()
    feats = torch.from_numpy(rng.standard_normal((rows, 16)).astype(np.float32)).cuda()
    points = torch.from_numpy(rng.uniform(0, 1, (500 + 400 * seed, 4)).astype(np.float32)).cuda()
    torch.manual_seed(seed)
    net = torch.nn.ModuleList([spnn.SparseConv3d(16, 32, 3, stride=2, padding=1, indice_key="d"), spnn.SubMConv3d(32, 32, 3),
                               spnn.SparseInverseConv3d(32, 16, 3, indice_key="d")]).cuda()
    voxelize = spnn.Voxelization([0.1, 0.1, 0.1], [0, 0, 0, 1, 1, 1], 5, 300 + 100 * seed).cuda()

    def run(distinct):
        x = feats.clone().requires_grad_(True)
        t = spnn.SparseTensor(x, idx, SPACE, 1, distinct=distinct)
        for layer in net:
            t = layer(t)
        grads = torch.autograd.grad(t.features.square().sum(), [x] + list(net.parameters()))
        return [t.features.detach(), t.indices] + list(grads) + list(voxelize(points))
    return run


@pytest.mark.parametrize("share", [False, True])
def test_threads_on_one_stream(gpu_handle, share):
    import torch
    import mluop_hip
    from mluop_hip import nn as spnn
    threads, rounds = 6, 8
    jobs = [make_job(s) for s in range(threads)]
    # (guard bands wait for the device behind every call, which would keep the threads apart)
    guard, mluop_hip.GUARD_BYTES = mluop_hip.GUARD_BYTES, 0
    spnn.share_row_maps(share)
    try:
        alone = [[job(d) for d in (False, True)] for job in jobs]
        torch.cuda.synchronize()
        problems = []
        gate = threading.Barrier(threads)

        def work(n):
            try:
                gate.wait(60)
                for r in range(rounds):
                    distinct = (n + r) % 2
                    for i, (got, want) in enumerate(zip(jobs[n](bool(distinct)), alone[n][distinct])):
                        if not torch.equal(got, want):
                            problems.append("thread %d, round %d: output %d differs" % (n, r, i))
            except Exception as e:  # noqa: BLE001 (reported by the main thread)
                problems.append("thread %d: %r" % (n, e))

        pool = [threading.Thread(target=work, args=(n,)) for n in range(threads)]
        for t in pool:
            t.start()
        for t in pool:
            t.join(100)
        assert not any(t.is_alive() for t in pool)
        torch.cuda.synchronize()
        assert not problems, problems[:5]
    finally:
        spnn.share_row_maps(False)
        mluop_hip.GUARD_BYTES = guard


def test_threads_on_one_stream_in_guard_mode(gpu_handle):
    """The same with buffers that come from Python: a call holds its handle while it takes the GIL."""
    import torch
    import mluop_hip
    assert mluop_hip.GUARD_BYTES > 0
    jobs = [make_job(s) for s in range(3)]
    alone = [job(False) for job in jobs]
    torch.cuda.synchronize()
    problems = []

    def work(n):
        try:
            for _ in range(3):
                for got, want in zip(jobs[n](False), alone[n]):
                    if not torch.equal(got, want):
                        problems.append("thread %d differs" % n)
        except Exception as e:  # noqa: BLE001
            problems.append("thread %d: %r" % (n, e))

    pool = [threading.Thread(target=work, args=(n,)) for n in range(3)]
    for t in pool:
        t.start()
    for t in pool:
        t.join(100)
    assert not any(t.is_alive() for t in pool)
    assert not problems, problems[:5]
