"""What SparseSequential may leave out: a ReLU goes into the convolution's store, and a nested network's rulebooks into
the plan of the outer one, only where the modules' own calls would do the same and nothing else.  (Decisions of
the host: no GPU.)"""
import pytest
import torch

from mluop_hip import nn as spnn


def pair():
    return spnn.SubMConv3d(16, 16, 3), torch.nn.ReLU()


def test_plain_modules():
    for conv in (spnn.SubMConv3d(16, 16, 3), spnn.SparseConv3d(16, 16, 3), spnn.SparseInverseConv3d(16, 16, 3, "a")):
        assert spnn._relu_in_store(conv, torch.nn.ReLU())


@pytest.mark.parametrize("which", [0, 1])
def test_a_compiled_module_is_called(which):
    modules = pair()
    modules[which].compile(backend="eager")
    assert not spnn._relu_in_store(*modules)


@pytest.mark.parametrize("owner,which", [(spnn.SubMConv3d, 0), (spnn._ConvBase, 0), (torch.nn.ReLU, 1)])
def test_a_class_with_another_forward_is_called(owner, which, monkeypatch):
    modules = pair()
    real = owner.forward
    monkeypatch.setattr(owner, "forward", lambda self, x: real(self, x))
    assert not spnn._relu_in_store(*modules)
    monkeypatch.undo()
    assert spnn._relu_in_store(*modules)


@pytest.mark.parametrize("which", [0, 1])
def test_a_module_with_a_call_or_forward_of_its_own_is_called(which, monkeypatch):
    modules = pair()
    own = type(modules[which])
    monkeypatch.setattr(own, "__call__", lambda self, x: torch.nn.Module.__call__(self, x), raising=False)
    assert not spnn._relu_in_store(*modules)
    monkeypatch.undo()
    modules[which].forward = lambda x: x
    assert not spnn._relu_in_store(*modules)


class Cached(spnn.SparseSequential):
    """A network with a way of its own to come to its rulebooks."""

    def plan(self, x):
        self.planned = getattr(self, "planned", 0) + 1
        return x


class Given(spnn.SubMConv3d):
    """A layer with a way of its own to come to its rulebook."""

    def _rulebook(self, x):
        return x.rulebooks["given"]


@pytest.mark.parametrize("how", ["class", "instance"])
@pytest.mark.parametrize("in_network", [False, True])
def test_a_layers_own_rulebook_is_asked_for(how, in_network, monkeypatch):
    monkeypatch.setattr(spnn._IndiceConv, "apply", staticmethod(lambda features, weight, rb, *a, **k: features + rb))
    x = empty_tensor()
    x.rulebooks["given"] = 3.0
    layer = Given(16, 16, 3) if how == "class" else spnn.SubMConv3d(16, 16, 3)
    if how == "instance":
        layer._rulebook = lambda x: x.rulebooks["given"]
    net = spnn.SparseSequential(layer) if in_network else layer
    assert torch.equal(net(x).features, x.features + 3.0)


def empty_tensor():
    return spnn.SparseTensor(torch.zeros(2, 16), torch.zeros(2, 4, dtype=torch.int32), (4, 4, 4), 1)


@pytest.mark.parametrize("depth", [1, 2])
def test_a_nested_networks_own_plan_is_called(depth):
    inner = Cached(spnn.SubMConv3d(16, 16, 3), torch.nn.ReLU())
    net = inner
    for _ in range(depth):
        net = spnn.SparseSequential(net)
    net.plan(empty_tensor())
    assert inner.planned == 1

    plain, seen = spnn.SparseSequential(torch.nn.ReLU()), []
    plain.plan = lambda x: (seen.append(x), x)[1]
    outer = spnn.SparseSequential(plain)
    x = empty_tensor()
    assert outer.plan(x) is x and seen == [x]
