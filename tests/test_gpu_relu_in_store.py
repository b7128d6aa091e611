"""mluOpExtSetForwardRelu: every gather kernel stores max(sum, 0) of the sums it stores without it, bit for bit, and
a SparseSequential that uses it gives the results and gradients of its layers called one by one."""
import numpy as np
import pytest

from spconv_cases import random_voxels
from test_gpu_pair_lists import kernels_of
from test_gpu_tall_tiles import make_case

pytestmark = pytest.mark.gpu

CHOICES = ("dense_tiles", "wave_per_tile", "tall_tiles", "gather_simt", "lists_on_trust")


@pytest.mark.parametrize("ci,co", [(64, 64), (4, 16), (16, 33), (128, 128)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("rows,shuffle", [(1, False), (1100, False), (1100, True)])
@pytest.mark.parametrize("on", ["dense_tiles", "wave_per_tile", "tall_tiles", "gather_simt", "none"])
@pytest.mark.parametrize("rulebook", ["lists", "maps", "twice"])
def test_sums_stored_without_their_negatives(gpu_handle, ci, co, dtype_name, rows, shuffle, on, rulebook):
    import torch
    import mluop_hip as m
    print("relu in store", ci, co, dtype_name, rows, shuffle, on, rulebook, flush=True)
    case = make_case(gpu_handle, rows, (9, 20, 20), (3, 3, 3), ci, co, dtype_name, shuffle)
    pairs = case["pairs"]
    if rulebook == "twice":  # every offset has its first pair twice: the row is rebuilt from the pair lists
        pairs = pairs.clone()
        for k, n in enumerate(case["num"]):
            if n > 1:
                pairs[k, :, 1] = pairs[k, :, 0]
    case["x"][0, 0] = float("nan")

    def forward():
        return m.indice_conv_forward(gpu_handle, case["x"], case["w"], m.LAYOUT_ARRAY, pairs, case["num"],
                                     case["n_out"], True)

    for which in CHOICES:
        gpu_handle.set_kernel_choice(which, which == on)
    if rulebook != "maps":
        gpu_handle.set_kernel_choice("lists_on_trust", None)
    try:
        plain, plain_ran = kernels_of(gpu_handle, forward)
        gpu_handle.set_forward_relu(True)
        stored, stored_ran = kernels_of(gpu_handle, forward)
        gpu_handle.set_forward_relu(False)
        again = forward()
    finally:
        gpu_handle.set_forward_relu(False)
        for which in CHOICES:
            gpu_handle.set_kernel_choice(which, None)
    torch.cuda.synchronize()
    assert plain_ran == stored_ran
    assert torch.equal(plain.isnan(), stored.isnan()) and torch.equal(plain.isnan(), again.isnan())
    plain, stored, again = (t.nan_to_num(7.0) for t in (plain, stored, again))
    assert torch.equal(stored, plain.relu()) and torch.equal(again, plain)
    if rows > 1:
        assert (plain < 0).any() and (stored == 0).any() and (stored > 0).any()


def layers_of(spnn, torch):
    relu = torch.nn.ReLU()
    return [spnn.SubMConv3d(16, 16, 3, indice_key="a"), relu, spnn.SubMConv3d(16, 32, 3, indice_key="a"), relu,
            spnn.SubMConv3d(32, 32, 3, bias=True), torch.nn.ReLU(),
            spnn.SparseConv3d(32, 64, 3, stride=2, padding=1, indice_key="down"), torch.nn.ReLU(),
            spnn.SparseSequential(spnn.SubMConv3d(64, 64, 3), torch.nn.ReLU()), torch.nn.ReLU(),
            spnn.SparseInverseConv3d(64, 16, 3, indice_key="down"), torch.nn.ReLU6(), spnn.SubMConv3d(16, 16, 3)]


@pytest.mark.parametrize("dtype_name", ["float16", "float32"])
@pytest.mark.parametrize("rows", [1, 900])
def test_the_layers_results_and_gradients(gpu_handle, dtype_name, rows):
    import torch
    from mluop_hip import nn as spnn
    torch.manual_seed(rows)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(rows), 1, (9, 20, 20), rows)).cuda()
    layers = layers_of(spnn, torch)
    net = spnn.SparseSequential(*layers).cuda()
    feats = torch.randn(rows, 16, device="cuda", dtype=getattr(torch, dtype_name))

    def run(call):
        x = feats.clone().requires_grad_(True)
        net.zero_grad()
        y = call(spnn.SparseTensor(x, idx, (9, 20, 20), 1, distinct=True)).features
        (y.float() * torch.linspace(-1, 1, y.numel(), device="cuda").view_as(y)).sum().backward()
        return [y.detach(), x.grad] + [p.grad.clone() for p in net.parameters()]

    def one_by_one(t):
        for m in layers[:8] + list(layers[8]) + layers[9:]:
            t = m(t) if isinstance(m, spnn._ConvBase) else t.replace_features(m(t.features))
        return t

    for a, b in zip(run(net), run(one_by_one)):
        assert torch.equal(a, b)


def test_who_watches_the_layers_sees_them(gpu_handle, monkeypatch):
    import torch
    from mluop_hip import nn as spnn
    idx = torch.from_numpy(random_voxels(np.random.default_rng(3), 1, (9, 20, 20), 300)).cuda()
    conv, relu = spnn.SubMConv3d(16, 16, 3), torch.nn.ReLU()
    net = spnn.SparseSequential(conv, relu).cuda().requires_grad_(False)
    x = torch.randn(300, 16, device="cuda")
    stored = []
    real = spnn._IndiceConv.apply
    monkeypatch.setattr(spnn._IndiceConv, "apply", lambda *a, **k: (stored.append(bool(k.get("relu"))), real(*a, **k))[1])

    def forward():
        stored.clear()
        y = net(spnn.SparseTensor(x, idx, (9, 20, 20), 1)).features
        return y, stored[:]

    ref, used = forward()
    assert used == [True]
    seen = []
    for m in (conv, relu):
        for register in (m.register_forward_hook, m.register_forward_pre_hook):
            hook = register(lambda *a: seen.append(type(a[0])))
            y, used = forward()
            hook.remove()
            assert used == [False] and seen == [type(m)] and torch.equal(y, ref)
            seen.clear()
    hook = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(type(a[0])))
    y, used = forward()
    hook.remove()
    assert used == [False] and seen == [spnn.SubMConv3d, torch.nn.ReLU, spnn.SparseSequential] and torch.equal(y, ref)

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    with Mode():
        y, used = forward()
    assert used == [False] and "relu" in seen and torch.equal(y, ref)
    assert forward()[1] == [True]
    relu.inplace = True  # guard bands (on in these tests) make the result a view: no store for autograd's refusal
    y, used = forward()[0].clone(), forward()[1]
    monkeypatch.setattr(spnn, "_guarded", lambda: False)
    assert used == [False] and torch.equal(y, ref)
    y, used = forward()
    assert used == [True] and torch.equal(y, ref)
