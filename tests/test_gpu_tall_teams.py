"""Tall tiles of 512 rows with two teams of multiplying waves (2-byte types, more than 32 offsets, rows of 33 channels
up): the bits of the pair-list kernel of short tiles at row counts around a tile, with offsets that fill whole
tiles, none and a few rows of them, and the fallback for lists that are not in order."""
import numpy as np
import pytest

from spconv_cases import check_close, from_torch, random_voxels
from test_gpu_pair_lists import kernels_of
from test_gpu_tall_tiles import both_directions, check, make_case
import sparse_conv_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co", [(64, 64), (48, 100), (128, 128), (65, 65)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("rows,space", [(1, (4, 4, 4)), (511, (8, 9, 10)), (512, (8, 8, 8)), (513, (40, 60, 60)),
                                        (2049, (12, 20, 24))])
def test_bits_of_the_short_tiles(gpu_handle, ci, co, dtype_name, rows, space):
    print("tall teams", ci, co, dtype_name, rows, flush=True)
    case = make_case(gpu_handle, rows, space, (3, 3, 5), ci, co, dtype_name, False)
    check(gpu_handle, case, (True, True))
    both_directions(gpu_handle, case, True)
    assert all("gatherConvTall512" in names for names in case["kernels"]), case["kernels"]


@pytest.mark.parametrize("ci,co,rows,forward,backward", [
    (64, 64, 65025, True, True),       # 128 workgroups
    (64, 64, 65024, False, False),     # 127
    (128, 64, 65025, True, True),      # two groups of columns backward
    (64, 128, 32600, True, False),     # 128 and 64 workgroups
    (64, 32, 65025, None, False),      # (results of up to 32 columns have another kernel; rows of 32 channels stay with 256)
])
def test_by_workgroups(gpu_handle, ci, co, rows, forward, backward):
    """Which tiles a layer of 45 offsets takes by itself, and the same bits with either."""
    import torch
    import mluop_hip as m
    print("tall teams by workgroups", ci, co, rows, flush=True)
    case = make_case(gpu_handle, rows, (20, 240, 240) if rows > 40000 else (20, 180, 180), (3, 3, 5), ci, co, "float16", False)
    assert 2.2 < sum(case["num"]) / rows < 4  # pairs a row
    got = {}
    for tall in (None, False):
        gpu_handle.set_kernel_choice("tall_tiles", tall)
        try:
            got[tall] = [kernels_of(gpu_handle, call) for call in (
                lambda: m.indice_conv_forward(gpu_handle, case["x"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"],
                                              rows, True),
                lambda: m.indice_conv_backward_data(gpu_handle, case["dy"], case["w"], m.LAYOUT_ARRAY, case["pairs"],
                                                    case["num"], True, ci))]
        finally:
            gpu_handle.set_kernel_choice("tall_tiles", None)
    for (a, names), (b, short), tall in zip(got[None], got[False], (forward, backward)):
        assert torch.equal(a, b) and "gatherConvTall512" not in short
        assert tall is None or ("gatherConvTall512" in names) == tall and ("gatherConvTall" in names) == (not tall), names


def test_lists_that_are_not_in_order(gpu_handle):
    import torch
    rows, space, ks, channels = 1100, (8, 16, 16), (3, 3, 5), 64
    case = make_case(gpu_handle, rows, space, ks, channels, channels, "float16", False)
    pairs = case["pairs"].cpu().numpy().copy()
    rng = np.random.default_rng(3)
    for k, n in enumerate(case["num"]):
        order = rng.permutation(n)
        pairs[k, :, :n] = pairs[k][:, :n][:, order]
    case["pairs"].copy_(torch.from_numpy(pairs))
    out, dx, ran = both_directions(gpu_handle, case, True)
    torch.cuda.synchronize()
    assert ran == (True, True) and all("gatherConvTall512" in names for names in case["kernels"])
    w_k = from_torch(case["w"]).reshape(45, channels, channels)
    ref = oracle.forward(case["host"]["x"], w_k, pairs, case["num"], case["n_out"])
    check_close(from_torch(out), ref, "float16", "tall teams")
    ref = oracle.backward_data(case["host"]["dy"], w_k, pairs, case["num"])
    check_close(from_torch(dx), ref, "float16", "tall teams")


def with_and_without_a_wait(handle, idx, space, ks, stride, x, w):
    """Forward on a rulebook whose report is there, and on one whose report is not: (result, kernels) of each.  Rows that are not
    in order run over the row map then, behind list kernels that were launched on trust and return."""
    import torch
    import mluop_hip as m
    sub_m = stride == 1
    pad = [k // 2 for k in ks]
    out_space = list(space) if sub_m else [(s + 2 * p - k) // stride + 1 for s, p, k in zip(space, pad, ks)]
    idx = torch.from_numpy(idx).cuda()

    def rulebook():
        return m.get_indice_pairs(handle, idx, 1, space, ks, out_space, pad, [stride] * 3, [1, 1, 1], sub_m)

    pairs, _, num, n_out = rulebook()
    torch.cuda.synchronize()
    num = [int(v) for v in num.cpu()]
    got = [kernels_of(handle, lambda: m.indice_conv_forward(handle, x, w, m.LAYOUT_ARRAY, pairs, num, n_out, sub_m))]
    torch.cuda.synchronize()
    guard_bytes, m.GUARD_BYTES = m.GUARD_BYTES, 0  # (checked after a wait)
    try:
        busy = torch.ones((4096, 4096), device="cuda")

        def call():
            a = busy
            for _ in range(40):  # some 40 milliseconds in front of the rulebook
                a = (a @ a) * 1e-4
            return m.indice_conv_forward(handle, x, w, m.LAYOUT_ARRAY, rulebook()[0], num, n_out, sub_m)
        got.append(kernels_of(handle, call))
        torch.cuda.synchronize()
    finally:
        m.GUARD_BYTES = guard_bytes
    return got, sum(num) / n_out / len(num)


def test_row_map_behind_lists_on_trust():
    """The row map's tiles are of 256 rows (5000 rows: more than a grid for 512, rounded up to eight tiles, covers)."""
    import torch
    import mluop_hip as m
    space, ks = (12, 24, 24), (3, 3, 5)
    rng = np.random.default_rng(8)
    idx = random_voxels(rng, 1, space, 5000, shuffle=True)
    x = torch.from_numpy(rng.standard_normal((5000, 64)).astype(np.float32)).cuda().half()
    w = torch.from_numpy((rng.standard_normal(ks + (64, 64)) / 50).astype(np.float32)).cuda().half()
    handle = m.make_handle_on_current_stream()
    handle.set_kernel_choice("dense_tiles", False)
    handle.set_kernel_choice("tall_tiles", True)
    ((want, known), (got, trusted)), _ = with_and_without_a_wait(handle, idx, space, ks, 1, x, w)
    assert "packFilterCutPairLists" not in known and "gatherConvTall" in known and "gatherConvTall512" not in known, known
    assert "packFilterCutPairLists" in trusted and "gatherConvTall512" in trusted and "gatherConvTall" in trusted, trusted
    assert torch.equal(got, want)
