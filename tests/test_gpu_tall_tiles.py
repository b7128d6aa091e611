"""The gather kernel of tall tiles: at row counts around its tiles of 256 (rows of 512 bytes: 512)
result rows, with lists that hold less and far more than one filling of its LDS, for pair lists and row
maps, in both directions.  It adds what the pair-list kernel of short tiles adds, in the same order, so
its results are held to that kernel's bits, and that kernel to the oracle by the other operator tests."""
import numpy as np
import pytest

from spconv_cases import check_close, from_torch, random_voxels, round_to, to_torch
from test_gpu_pair_lists import gpu_rulebook, kernels_of
import sparse_conv_oracle as oracle

pytestmark = pytest.mark.gpu


def both_directions(handle, case, tall):
    import mluop_hip as m
    handle.set_kernel_choice("dense_tiles", False)
    handle.set_kernel_choice("wave_per_tile", False)
    handle.set_kernel_choice("tall_tiles", tall)
    try:
        out, forward = kernels_of(handle, lambda: m.indice_conv_forward(
            handle, case["x"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"], case["n_out"], case["sub_m"]))
        dx, backward = kernels_of(handle, lambda: m.indice_conv_backward_data(
            handle, case["dy"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"], case["sub_m"], case["ci"]))
    finally:
        for which in ("dense_tiles", "wave_per_tile", "tall_tiles"):
            handle.set_kernel_choice(which, None)
    case["kernels"] = forward, backward
    return out, dx, tuple("gatherConvTall" in names or "gatherConvTall512" in names for names in case["kernels"])


def make_case(handle, rows, space, ks, ci, co, dtype_name, shuffle, stride=1):
    rng = np.random.default_rng(rows + ci)
    idx = random_voxels(rng, 1, space, rows, shuffle=shuffle)
    sub_m = stride == 1
    pairs, num, n_out = gpu_rulebook(handle, idx, 1, space, ks, [k // 2 for k in ks], [stride] * 3, [1, 1, 1], sub_m)
    K = int(np.prod(ks))
    b = 1.0 / np.sqrt(K * ci)
    host = dict(x=round_to(rng.standard_normal((idx.shape[0], ci)).astype(np.float32), dtype_name),
                w=round_to(rng.uniform(-b, b, tuple(ks) + (ci, co)).astype(np.float32), dtype_name),
                dy=round_to((rng.standard_normal((n_out, co)) * 0.1).astype(np.float32), dtype_name))
    case = {k: to_torch(v, dtype_name, "cuda") for k, v in host.items()}
    case.update(pairs=pairs, num=num, n_out=n_out, sub_m=sub_m, ci=ci, host=host)
    return case


def check(handle, case, wide):
    import torch
    out, dx, ran = both_directions(handle, case, True)
    ref_out, ref_dx, _ = both_directions(handle, case, False)
    torch.cuda.synchronize()
    assert ran == wide, ran
    assert torch.equal(out, ref_out) and torch.equal(dx, ref_dx)


@pytest.mark.parametrize("ci,co", [(64, 64), (5, 128), (16, 33), (48, 100), (128, 64), (65, 65)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("rows,space", [(1, (4, 4, 4)), (255, (9, 20, 20)), (256, (8, 8, 8)), (257, (9, 20, 20)),
                                        (513, (8, 9, 10)), (1100, (8, 12, 12))])
@pytest.mark.parametrize("shuffle", [False, True])
def test_bits_of_the_short_tiles(gpu_handle, ci, co, dtype_name, rows, space, shuffle):
    print("tall tiles", ci, co, dtype_name, rows, shuffle, flush=True)
    case = make_case(gpu_handle, rows, space, (3, 3, 3), ci, co, dtype_name, shuffle)
    check(gpu_handle, case, (co > 32, ci > 32))


@pytest.mark.parametrize("ks,stride,rows,space", [
    ((5, 5, 5), 1, 900, (10, 12, 12)),      # more offsets than lanes; several fillings of the lists a tile
    ((5, 5, 5), 1, 600, (30, 40, 40)),      # ... most of them without a pair
    ((5, 5, 7), 1, 400, (10, 10, 10)),      # more than 128 offsets: row map, counts in device memory
    ((2, 2, 2), 2, 700, (16, 16, 16)),
    ((3, 3, 3), 2, 700, (16, 24, 24)),
])
@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 64, 128), ("float32", 128, 64), ("bfloat16", 128, 128)])
@pytest.mark.parametrize("shuffle", [False, True])
def test_other_kernels_and_strides(gpu_handle, ks, stride, rows, space, dtype_name, ci, co, shuffle):
    print("tall tiles", ks, stride, rows, dtype_name, ci, co, shuffle, flush=True)
    check(gpu_handle, make_case(gpu_handle, rows, space, ks, ci, co, dtype_name, shuffle, stride), (True, True))


@pytest.mark.parametrize("dtype_name,channels", [("float16", 64), ("float32", 128)])
def test_lists_out_of_order_and_filters_that_are_not_finite(gpu_handle, dtype_name, channels):
    """The pair tensor is written over with a shuffled rulebook's: every tile collects its pairs by reading
    all of them.  And an infinite filter reaches the rows with a pair at its offset only."""
    import torch
    rows, space, ks = 700, (8, 16, 16), (3, 3, 3)
    case = make_case(gpu_handle, rows, space, ks, channels, channels, dtype_name, False)
    case["w"][0, 1, 2, 3, 4] = float("inf")
    w_k = from_torch(case["w"]).reshape(27, channels, channels)
    x, dy = case["host"]["x"], case["host"]["dy"]

    def graded(pairs_np):
        out, dx, ran = both_directions(gpu_handle, case, True)
        torch.cuda.synchronize()
        assert ran == (True, True)
        for got, ref in ((from_torch(out), oracle.forward(x, w_k, pairs_np, case["num"], case["n_out"])),
                         (from_torch(dx), oracle.backward_data(dy, w_k, pairs_np, case["num"]))):
            finite = np.isfinite(ref)
            assert np.array_equal(np.isfinite(got), finite) and not finite.all()
            check_close(got[finite], ref[finite], dtype_name, "tall tiles")

    graded(case["pairs"].cpu().numpy())
    rng = np.random.default_rng(3)
    idx = random_voxels(np.random.default_rng(rows + channels), 1, space, rows, shuffle=False)
    rp, _, rn, _ = oracle.get_indice_pairs(np.ascontiguousarray(idx[rng.permutation(rows)]), 1, [1, 1, 1], [1, 1, 1],
                                           [1, 1, 1], list(ks), list(space), True)
    assert [int(v) for v in rn] == case["num"]
    for k in range(27):   # (the input rows out of order too, so that both directions meet lists that cannot be cut)
        rp[k, :, :rn[k]] = rp[k][:, rng.permutation(rn[k])]
    case["pairs"].copy_(torch.from_numpy(rp).cuda())
    graded(rp)
