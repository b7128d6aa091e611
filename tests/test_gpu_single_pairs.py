"""The promise that a pair column names every row once (mluOpExtSetSinglePairsPromise): the same numbers as without it,
for the gradient of a strided layer's input and for the inverse layer's result, and who makes it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# kernel and stride; in the last two, rows are in no pair
SHAPES = [((2, 2, 2), (2, 2, 2)), ((1, 1, 1), (1, 1, 1)), ((2, 3, 1), (2, 3, 1)), ((1, 1, 1), (2, 2, 2)),
          ((2, 1, 2), (3, 2, 2))]


def rulebook(handle, rows, ks, stride, repeated=False):
    import torch
    import mluop_hip as m
    rng = np.random.default_rng(rows + ks[0])
    space = (9, 21, 31)
    cells = rng.choice(space[0] * space[1] * space[2], rows, replace=repeated)
    if rows == 1:
        cells[:] = 0  # (whatever the stride, some output reaches the first cell)
    idx = np.stack([0 * cells, cells // (21 * 31), cells // 31 % 21, cells % 31], axis=1).astype(np.int32)
    out = [(s - k) // t + 1 for s, k, t in zip(space, ks, stride)]
    pairs, _, num, n_out = m.get_indice_pairs(handle, torch.from_numpy(idx).cuda(), 1, space, ks, out, [0, 0, 0],
                                              list(stride), [1, 1, 1], False)
    return pairs, [int(v) for v in num.cpu()], n_out


@pytest.mark.parametrize("rows", [1, 63, 65, 1000, 5000])
@pytest.mark.parametrize("ks,stride", SHAPES)
@pytest.mark.parametrize("dtype_name,q,c", [("float16", 16, 16), ("float16", 128, 128), ("bfloat16", 64, 33), ("float16", 5, 17),
                                            ("bfloat16", 24, 96), ("float32", 64, 96), ("float32", 128, 64),
                                            ("float32", 100, 128), ("float32", 16, 5), ("float32", 32, 32)])
@pytest.mark.parametrize("inverse", [False, True])
def test_same_numbers_as_without_the_promise(gpu_handle, rows, ks, stride, dtype_name, q, c, inverse):
    import torch
    import mluop_hip as m
    print("single pairs", rows, ks, stride, dtype_name, q, c, inverse, flush=True)
    pairs, counts, n_out = rulebook(gpu_handle, rows, ks, stride, repeated=rows == 1000 and max(ks) > 1)
    assert n_out > 0
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((n_out, q), generator=g, device="cuda").to(dtype)
    ci, co = (q, c) if inverse else (c, q)
    w = torch.randn(tuple(ks) + (ci, co), generator=g, device="cuda").to(dtype)

    def run():
        if inverse:
            return m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, rows, False, inverse=1)
        return m.indice_conv_backward_data(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, False, ci)
    gpu_handle.set_extended_modes(True)
    try:
        ref = run()
        gpu_handle.promise_single_pairs(0)
        gpu_handle.set_kernel_timing(True)
        got = run()
        names = [n for n, _ in gpu_handle.kernel_timings()]
        gpu_handle.set_kernel_timing(False)
    finally:
        gpu_handle.promise_single_pairs(None)
        gpu_handle.set_extended_modes(False)
    assert "gatherConvSingle" in names, names
    k = w.reshape(-1, ci, co).double()
    want = torch.zeros((rows, c), dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    for o, n in enumerate(counts):
        i, j = pairs[o, 0, :n].long(), pairs[o, 1, :n].long()
        f = k[o] if inverse else k[o].T
        want.index_add_(0, i, x[j].double() @ f)
        size.index_add_(0, i, x[j].double().abs() @ f.abs())
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    bound = 2.0 ** -24 * q * size + rounding * want.abs() + (2.0 ** -25 if dtype_name == "float16" else 0)
    assert ((got.double() - want).abs() <= bound).all()
    assert ((ref.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("dtype_name,q,c", [("float16", 64, 96), ("float32", 40, 24), ("bfloat16", 128, 128)])
@pytest.mark.parametrize("finite", [True, False])
def test_partners_out_of_range_give_zero_rows(gpu_handle, dtype_name, q, c, finite, relu):
    """Every row is in a pair, so that nothing clears the result, and some pairs' other row does not exist.  (The
    kernel looks at every index before it uses it.)"""
    import torch
    import mluop_hip as m
    rows, ks, stride = 1500, (1, 1, 1), (1, 1, 1)
    pairs, counts, n_out = rulebook(gpu_handle, rows, ks, stride)
    assert counts == [rows] and n_out == rows
    out_of_range = {3: -1, 64: n_out, 200: 1 << 30, 1499: -(1 << 31)}
    for at, value in out_of_range.items():
        pairs[0, 1, at] = value
    bad = pairs[0, 0, list(out_of_range)].long()
    dtype = getattr(torch, dtype_name)
    x = torch.randn((n_out, q), device="cuda").to(dtype)
    w = torch.randn((1, 1, 1, q, c), device="cuda").to(dtype)
    if not finite:
        w[0, 0, 0, 5, 7], w[0, 0, 0, 6, 1] = float("inf"), float("nan")
    gpu_handle.set_extended_modes(True)
    gpu_handle.promise_single_pairs(0)
    gpu_handle.set_forward_relu(relu)
    try:
        torch.full((rows, c), 7.0, device="cuda", dtype=dtype)  # (what the allocator hands out next is not zero)
        got = m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, rows, False, inverse=1)
    finally:
        gpu_handle.set_forward_relu(False)
        gpu_handle.promise_single_pairs(None)
        gpu_handle.set_extended_modes(False)
    assert (got[bad] == 0).all()
    good = torch.ones(rows, dtype=torch.bool, device="cuda")
    good[bad] = False
    partner = torch.zeros(rows, dtype=torch.int64, device="cuda")
    keep = good[pairs[0, 0].long()]
    partner[pairs[0, 0].long()[keep]] = pairs[0, 1].long()[keep]
    want = x[partner].double() @ w[0, 0, 0].double()
    want = want.clamp(min=0) if relu else want
    size = x[partner].double().abs() @ w[0, 0, 0].double().abs()
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    ok = (got.double() - want).abs() <= 2.0 ** -24 * q * size + rounding * want.abs() + 2.0 ** -25
    same = (got.double() == want) | (got.isnan() & want.isnan())  # (infinities and NaN)
    assert (ok | same)[good].all()


def test_relu_in_the_store(gpu_handle):
    import torch
    import mluop_hip as m
    pairs, counts, n_out = rulebook(gpu_handle, 700, (1, 1, 1), (2, 2, 2))
    x = torch.randn((n_out, 64), device="cuda").half()
    w = torch.randn((1, 1, 1, 64, 64), device="cuda").half()
    gpu_handle.set_extended_modes(True)
    gpu_handle.promise_single_pairs(0)
    try:
        plain = m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, 700, False, inverse=1)
        gpu_handle.set_forward_relu(True)
        got = m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, 700, False, inverse=1)
    finally:
        gpu_handle.set_forward_relu(False)
        gpu_handle.promise_single_pairs(None)
        gpu_handle.set_extended_modes(False)
    assert torch.equal(got, plain.clamp(min=0)) and (plain < 0).any()


@pytest.mark.parametrize("backward", [False, True])
@pytest.mark.parametrize("dtype_name,q,c", [("float16", 64, 64), ("bfloat16", 33, 128), ("float32", 48, 20)])
def test_the_other_column(gpu_handle, backward, dtype_name, q, c):
    """Column 1 names the rows of a plain layer's result and of an inverse layer's gradient; calls whose result rows the
    other column names stay with the ordinary kernels."""
    import torch
    import mluop_hip as m
    rows, ks, stride = 900, (1, 1, 1), (1, 1, 1)
    pairs, counts, n_out = rulebook(gpu_handle, rows, ks, stride)
    dtype = getattr(torch, dtype_name)
    x = torch.randn((rows, q), device="cuda").to(dtype)
    w = torch.randn((1, 1, 1) + ((c, q) if backward else (q, c)), device="cuda").to(dtype)

    def run(other=False):
        # the layer and its inverse: which of them has its result rows in column 1 depends on the direction
        inverse = int(backward != other)
        gpu_handle.set_kernel_timing(True)
        if backward:
            y = m.indice_conv_backward_data(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, False, c, inverse=inverse,
                                            rows=rows)
        else:
            y = m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, rows, False, inverse=inverse)
        torch.cuda.synchronize()
        names = [n for n, _ in gpu_handle.kernel_timings()]
        gpu_handle.set_kernel_timing(False)
        return y, names
    gpu_handle.set_extended_modes(True)
    try:
        ref, plain = run()
        gpu_handle.promise_single_pairs(1)
        got, names = run()
        _, others = run(other=True)
    finally:
        gpu_handle.promise_single_pairs(None)
        gpu_handle.set_extended_modes(False)
    assert "gatherConvSingle" in names and "gatherConvSingle" not in plain + others, (names, plain, others)
    want = torch.zeros((rows, c), dtype=torch.float64, device="cuda")
    f = w[0, 0, 0].double().T if backward else w[0, 0, 0].double()
    source = pairs[0, 0].long()
    want[pairs[0, 1].long()] = x[source].double() @ f
    size = torch.zeros_like(want)
    size[pairs[0, 1].long()] = x[source].double().abs() @ f.abs()
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    bound = 2.0 ** -24 * q * size + rounding * want.abs() + 2.0 ** -25
    assert ((got.double() - want).abs() <= bound).all() and ((ref.double() - want).abs() <= bound).all()


def test_layers_promise_what_their_geometry_says():
    import torch
    from mluop_hip import nn as spnn
    rng = np.random.default_rng(0)
    cells = rng.choice(8 * 16 * 16, 500, replace=False)
    idx = np.stack([0 * cells, cells // 256, cells // 16 % 16, cells % 16], axis=1).astype(np.int32)
    x = spnn.SparseTensor(torch.randn((500, 16), device="cuda"), torch.from_numpy(idx).cuda(), (8, 16, 16), 1, distinct=True)
    for layer, single in ((spnn.SparseConv3d(16, 16, 2, stride=2, indice_key="a"), True),
                          (spnn.SparseConv3d(16, 16, 3, stride=2, padding=1, indice_key="b"), False),
                          (spnn.SparseConv3d(16, 16, 2, dilation=2, indice_key="c"), False),
                          (spnn.SparseConv3d(16, 16, 1, indice_key="d"), True),
                          (spnn.SubMConv3d(16, 16, 1, indice_key="e"), False)):
        y = layer.cuda()(x)
        assert x.rulebooks[layer.indice_key].single == single
        if not layer.sub_m:
            up = spnn.SparseInverseConv3d(16, 16, layer.kernel_size, layer.indice_key).cuda()
            assert up(y).features.shape == (500, 16)
    handle = spnn._handle()
    import ctypes
    import mluop_hip as m
    column = ctypes.c_int(7)
    m.check(m.lib().mluOpExtGetSinglePairsPromise(handle.ptr, ctypes.byref(column)))
    assert column.value == -1   # (a layer's call leaves the setting as it was)
