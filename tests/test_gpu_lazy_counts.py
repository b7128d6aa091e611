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
def test_counts_that_are_copied_wait_for_no_other_stream(monkeypatch, asked_by, why):
    """(Streams share four hardware queues, and behind another stream's work in one of them everybody waits: so with several
    streams in turn, and one that goes on behind the counts is enough.)"""
    import torch
    import mluop_hip
    from mluop_hip import nn as spnn
    monkeypatch.setattr(mluop_hip, "GUARD_BYTES", 0)  # (guards are checked after a wait for the device)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(3), 1, SPACE, 500)).cuda()
    features = torch.randn(500, 8, device="cuda")
    size = 9 if why == "too many offsets" else 3  # (the handle keeps 343 counts of a rulebook)
    layer = spnn.SubMConv3d(8, 16, size).cuda()
    a = torch.ones(4096, 4096, device="cuda")
    with torch.no_grad():
        want = layer(spnn.SparseTensor(features, idx, SPACE, 1, distinct=True)).features
        for attempt in range(12):
            x = spnn.SparseTensor(features, idx, SPACE, 1, distinct=True)
            rb = pending(layer, x)
            if why == "no longer on file":
                for _ in range(40):
                    pending(spnn.SubMConv3d(8, 16, 3), spnn.SparseTensor(features, idx, SPACE, 1, distinct=True))
            torch.cuda.synchronize()
            busy = torch.cuda.Stream()
            with torch.cuda.stream(busy):
                for _ in range(200):  # about 1 ms each
                    a @ a
                done = busy.record_event()
            if asked_by == "operator":
                got = layer(x).features
            else:
                assert rb.indice_num[size ** 3 // 2] == 500
            went_on = not done.query()
            torch.cuda.synchronize()
            assert asked_by == "python" or torch.equal(got, want)
            print("attempt", attempt, "the other stream is still busy:", went_on, flush=True)
            if went_on:
                return
    raise AssertionError("waited for streams that have nothing to do with the rulebook")


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


def watch(seen):
    """Notes copies to the host and layers' results in the order in which they are made."""
    import torch
    from torch.utils._python_dispatch import TorchDispatchMode

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            result = func(*args, **(kwargs or {}))
            if isinstance(result, torch.Tensor):
                if result.device.type == "cpu" and isinstance(args[0], torch.Tensor) and args[0].is_cuda:
                    seen.append("copy")
                elif func is torch.ops.aten.empty.memory_format and result.dtype == torch.float32:
                    seen.append("result")
            return result
    return Watch()


def many_layers(layers, form, size=lambda i: 3):
    import torch
    from mluop_hip import nn as spnn
    torch.manual_seed(0)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(1), 1, SPACE, 900)).cuda()
    feats = torch.randn(900, 8, device="cuda")
    convs = [spnn.SubMConv3d(8, 8, size(i)).cuda() for i in range(layers)]
    inner = type("Inner", (Planned, spnn.SparseSequential), {}) if form.endswith("own") else spnn.SparseSequential
    net = spnn.SparseSequential(*convs) if form == "flat" else spnn.SparseSequential(*convs[:5], inner(*convs[5:]))
    return net, convs, feats, lambda: spnn.SparseTensor(feats, idx, SPACE, 1, distinct=True)


class Planned:
    """A network's own plan (put in front of SparseSequential below)."""

    def plan(self, x):
        return super().plan(x)


@pytest.mark.parametrize("layers", [11, 33, 40])
@pytest.mark.parametrize("form", ["flat", "nested", "nested with a plan of its own"])
def test_networks_of_many_rulebooks_copy_no_counts(layers, form):
    """A handle keeps the counts of 32 rulebooks: they are all taken before they leave."""
    import torch
    net, convs, feats, tensor = many_layers(layers, form)
    seen = []
    with torch.no_grad():
        want = tensor()
        for conv in convs:
            want = conv(want)
        torch.cuda.synchronize()
        with watch(seen):
            assert torch.ones(3, device="cuda").cpu().shape == (3,) and "copy" in seen  # (it sees them)
            seen.clear()
            got = net(tensor())
    assert "copy" not in seen and seen.count("result") == layers, seen
    assert torch.equal(got.features, want.features)


def test_counts_of_many_offsets_are_copied_in_front_of_the_convolutions():
    import torch
    net, convs, feats, tensor = many_layers(6, "flat", lambda i: 9 if i % 2 else 3)
    seen = []
    with torch.no_grad(), watch(seen):
        net(tensor())
    assert seen == ["copy"] * 3 + ["result"] * 6


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
