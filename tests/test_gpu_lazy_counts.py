"""Layers take a rulebook's pair counts when they run: when the handle has them on file no longer, on another
stream than the rulebook's, and from several threads at once."""
import threading

import numpy as np
import pytest

from spconv_cases import random_voxels

pytestmark = pytest.mark.gpu

SPACE = (9, 40, 40)


def setup(rows, seed=0):
    import torch
    from mluop_hip import nn as spnn
    torch.manual_seed(seed)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(seed), 1, SPACE, rows)).cuda()
    layer = spnn.SubMConv3d(8, 16, 3, indice_key="k").cuda()
    x = spnn.SparseTensor(torch.randn(rows, 8, device="cuda", requires_grad=True), idx, SPACE, 1, distinct=True)
    waited = spnn.SparseTensor(x.features, idx, SPACE, 1, distinct=True)
    assert isinstance(layer._rulebook(waited)._indice_num, list)
    want = layer(waited).features
    grads = torch.autograd.grad(want.sum(), [x.features, layer.weight])
    torch.cuda.synchronize()
    return layer, x, want.detach(), grads


def pending(layer, x):
    import torch
    rb = layer._rulebook(x, wait_counts=False)
    assert isinstance(rb._indice_num, torch.Tensor)
    return rb


def check(layer, x, want, grads):
    import torch
    y = layer(x).features
    assert torch.equal(y, want)
    for g, w in zip(torch.autograd.grad(y.sum(), [x.features, layer.weight]), grads):
        assert torch.equal(g, w)


@pytest.mark.parametrize("rows", [1, 700, 6000])
@pytest.mark.parametrize("others", [0, 40])
def test_counts_taken_by_the_operator(rows, others):
    from mluop_hip import nn as spnn
    layer, x, want, grads = setup(rows)
    rb = pending(layer, x)
    more = [pending(spnn.SubMConv3d(8, 16, 3).cuda(),
                    spnn.SparseTensor(x.features, x.indices, SPACE, 1, distinct=True)) for _ in range(others)]
    check(layer, x, want, grads)
    assert rb.indice_num[13] == rows and all(r.indice_num == rb.indice_num for r in more)


def test_on_another_stream():
    import torch
    layer, x, want, grads = setup(3000)
    pending(layer, x)
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        check(layer, x, want, grads)
    torch.cuda.current_stream().wait_stream(other)


@pytest.mark.parametrize("asked_by", ["operator", "python"])
@pytest.mark.parametrize("why", ["too many offsets", "no longer on file"])
def test_counts_that_are_copied_wait_for_no_other_stream(asked_by, why):
    import torch
    from mluop_hip import nn as spnn
    idx = torch.from_numpy(random_voxels(np.random.default_rng(3), 1, SPACE, 500)).cuda()
    x = spnn.SparseTensor(torch.randn(500, 8, device="cuda"), idx, SPACE, 1, distinct=True)
    size = 9 if why == "too many offsets" else 3  # (the handle keeps 343 counts of a rulebook)
    layer = spnn.SubMConv3d(8, 16, size).cuda()
    with torch.no_grad():
        want = layer(spnn.SparseTensor(x.features, idx, SPACE, 1, distinct=True)).features
        rb = pending(layer, x)
        if why == "no longer on file":
            for _ in range(40):
                pending(spnn.SubMConv3d(8, 16, 3), spnn.SparseTensor(x.features, idx, SPACE, 1, distinct=True))
        torch.cuda.synchronize()
        a, busy = torch.ones(4096, 4096, device="cuda"), torch.cuda.Stream()
        busy.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(busy):
            for _ in range(200):  # about 1 ms each
                b = a @ a
            done = busy.record_event()
        if asked_by == "operator":
            got = layer(x).features
        else:
            assert rb.indice_num[size ** 3 // 2] == 500
        assert not done.query(), "waited for a stream that has nothing to do with the rulebook"
        assert asked_by == "python" or torch.equal(got, want)
        torch.cuda.synchronize()
        del b


def test_counts_that_an_operator_took_are_not_asked_for_again():
    """Neither behind other rulebooks' nor while a graph is captured, which allows no wait."""
    import torch
    from mluop_hip import nn as spnn
    layer, x, want, grads = setup(3000)
    rb = pending(layer, x)
    check(layer, x, want, grads)
    for _ in range(40):
        pending(spnn.SubMConv3d(8, 16, 3), spnn.SparseTensor(x.features, x.indices, SPACE, 1, distinct=True))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pairs = rb.pairs
    counts = rb.indice_num
    assert counts[13] == 3000 and isinstance(counts, list)
    for _ in range(3):
        pairs.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert all((p[:, n:] == -1).all() and (p[:, :n] == 7).all() for p, n in zip(pairs, counts))


def test_from_several_threads():
    import torch
    for seed in range(5):
        layer, x, want, grads = setup(2500, seed)
        pending(layer, x)
        main = torch.cuda.current_stream()
        streams = [torch.cuda.Stream() for _ in range(3)] + [main]
        errors = []

        def work(stream):
            try:
                with torch.cuda.stream(stream):
                    if stream is not main:
                        stream.wait_stream(main)
                    for _ in range(3):
                        assert torch.equal(layer(x).features.detach(), want)
            except Exception as e:  # noqa: BLE001
                errors.append(e)
        threads = [threading.Thread(target=work, args=(s,)) for s in streams]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not errors, errors
