"""mluOpExtSetPairTails: without the -1 behind each offset's pairs the lists, counts and output rows are the same,
for every probe kernel and both row orders, and the next rulebook has its -1 again."""
import numpy as np
import pytest

from spconv_cases import out_space, random_voxels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks,stride,dilation,sub_m", [((3, 3, 3), 1, 1, True), ((5, 5, 5), 1, 1, True), ((3, 1, 7), 1, 1, True),
                                                      ((3, 3, 3), 1, 2, False), ((3, 3, 3), 2, 1, False),
                                                      ((2, 2, 2), 2, 1, False), ((3, 3, 1), 2, 1, False),
                                                      ((3, 3, 3), 1, 1, False)])
@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("rows", [1, 64, 1300])
def test_lists_without_tails(gpu_handle, ks, stride, dilation, sub_m, shuffle, rows):
    import torch
    import mluop_hip as m
    print("pair tails", ks, stride, dilation, sub_m, shuffle, rows, flush=True)
    space = (9, 18, 20)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(rows), 1, space, rows, shuffle=shuffle)).cuda()
    pad = [dilation * (k // 2) for k in ks]
    dil = [dilation] * 3
    ospace = list(space) if sub_m else out_space(space, ks, pad, [stride] * 3, dil)

    def build(**kwargs):
        return m.get_indice_pairs(gpu_handle, idx, 1, space, ks, ospace, pad, [stride] * 3, dil, sub_m, **kwargs)

    pairs, rows_out, num, n_out = build()
    bare, bare_rows, bare_num, bare_n = build(tails=False)
    again = build()
    assert torch.equal(num, bare_num) and n_out == bare_n and torch.equal(rows_out, bare_rows)
    for k, n in enumerate(num.cpu().tolist()):
        assert torch.equal(pairs[k, :, :n], bare[k, :, :n])
        assert (pairs[k, :, n:] == -1).all() and torch.equal(pairs[k], again[0][k])


@pytest.mark.parametrize("own", [0, 1])
def test_the_callers_settings_outlive_a_call(gpu_handle, own):
    """A call and a layer that change a setting of the handle for themselves leave it as the caller had it."""
    import ctypes
    import torch
    import mluop_hip as m
    from mluop_hip import nn as spnn
    lib, space, rows = m.lib(), (9, 18, 20), 500
    idx = torch.from_numpy(random_voxels(np.random.default_rng(3), 1, space, rows, shuffle=False)).cuda()

    def setting(handle, get):
        value = ctypes.c_int(-1)
        m.check(get(handle.ptr, ctypes.byref(value)))
        return value.value

    def build(handle, **kwargs):
        return m.get_indice_pairs(handle, idx, 1, space, (3, 3, 3), space, [1] * 3, [1] * 3, [1] * 3, True, **kwargs)

    m.check(lib.mluOpExtSetPairTails(gpu_handle.ptr, own))
    try:
        build(gpu_handle, tails=False)
        assert setting(gpu_handle, lib.mluOpExtGetPairTails) == own
        with pytest.raises(m.MluOpError):  # (output space of another size: refused)
            m.get_indice_pairs(gpu_handle, idx, 1, space, (3, 3, 3), (9, 18, 21), [1] * 3, [1] * 3, [1] * 3, True,
                               out_rows=rows, tails=False)
        assert setting(gpu_handle, lib.mluOpExtGetPairTails) == own
    finally:
        m.check(lib.mluOpExtSetPairTails(gpu_handle.ptr, 1))

    handle = spnn._handle()  # the layers' own: what is set on it does not reach into a layer without a ReLU
    conv = spnn.SubMConv3d(16, 16, 3).cuda()
    x = spnn.SparseTensor(torch.randn(rows, 16, device="cuda"), idx, space, 1, distinct=True)
    with torch.no_grad():
        plain = conv(x).features
        handle.set_forward_relu(own)
        try:
            assert torch.equal(conv(x).features, plain)
            assert torch.equal(spnn.SparseSequential(conv, torch.nn.ReLU())(x).features, plain.relu())
            assert setting(handle, lib.mluOpExtGetForwardRelu) == own
        finally:
            handle.set_forward_relu(False)


@pytest.mark.parametrize("layer,rows", [("subm", 1), ("subm", 1300), ("strided", 700), ("network", 900)])
@pytest.mark.parametrize("inference", [False, True])
def test_the_pairs_of_a_layers_rulebook(gpu_handle, layer, rows, inference):
    """Whoever asks a layer's rulebook for its pairs finds -1 behind them, as in the operator's own result."""
    import torch
    import mluop_hip as m
    from mluop_hip import nn as spnn
    print("layer's pairs", layer, rows, inference, flush=True)
    space, ks = (9, 18, 20), 3
    idx = torch.from_numpy(random_voxels(np.random.default_rng(rows), 1, space, rows, shuffle=True)).cuda()
    conv = (spnn.SparseConv3d(16, 16, ks, stride=2, padding=1, indice_key="a") if layer == "strided"
            else spnn.SubMConv3d(16, 16, ks, indice_key="a"))
    net = (spnn.SparseSequential(conv, torch.nn.ReLU()) if layer == "network" else conv).cuda()
    sub_m = layer != "strided"
    ospace = list(space) if sub_m else out_space(space, [ks] * 3, [1] * 3, [2] * 3, [1] * 3)
    want, _, num, _ = m.get_indice_pairs(gpu_handle, idx, 1, space, [ks] * 3, ospace, [1] * 3, [1 if sub_m else 2] * 3,
                                         [1] * 3, sub_m)
    poison = [torch.full((27, 2, rows), 7, dtype=torch.int32, device="cuda") for _ in range(4)]
    torch.cuda.synchronize()
    del poison   # (so that the layer's tensor is one that held something else)
    with torch.inference_mode(inference):
        x = spnn.SparseTensor(torch.randn(rows, 16, device="cuda"), idx, space, 1, distinct=True)
        first = net(x).features
    rb = x.rulebooks["a"]
    assert rb.indice_num == [int(n) for n in num.cpu()]
    assert torch.equal(rb.pairs, want)
    with torch.no_grad():
        assert torch.equal(net(x).features, first)


def test_the_pairs_of_a_layers_rulebook_under_capture(gpu_handle):
    """First asked for while a graph is captured: no copy from the host, and set for eager readers all the same."""
    import torch
    from mluop_hip import nn as spnn
    space, rows = (9, 18, 20), 600
    idx = torch.from_numpy(random_voxels(np.random.default_rng(8), 1, space, rows, shuffle=True)).cuda()
    x = spnn.SparseTensor(torch.randn(rows, 16, device="cuda"), idx, space, 1, distinct=True)
    rulebooks = []
    for key in "ab":
        spnn.SubMConv3d(16, 16, 3, indice_key=key).cuda()(x)
        rulebooks.append(x.rulebooks[key])
    torch.cuda.synchronize()
    want = rulebooks[0].pairs.clone()
    rulebooks[1]._pairs[:, :, -1] = torch.where(want[:, :, -1] == -1, 7, want[:, :, -1])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        seen = rulebooks[1].pairs + 1
    assert torch.equal(rulebooks[1].pairs, want)
    for _ in range(3):
        seen.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(seen - 1, want)
