"""The dense gather kernel for rows above 64 bytes at the edges of its tiles, of its waves' shares and of its phases:
against the oracle, on pair lists and on row maps."""
import numpy as np
import pytest

import sparse_conv_oracle as oracle
from spconv_cases import check_close, from_torch, random_voxels, round_to, to_torch

pytestmark = pytest.mark.gpu

SPACE = (7, 11, 13)


# rows: groups of 16, tiles of 128; kernels of one offset, of an even and an odd number, of several chunks of 27
@pytest.mark.parametrize("rows", [1, 16, 17, 127, 129, 400])
@pytest.mark.parametrize("ks", [(1, 1, 1), (1, 1, 2), (3, 3, 3), (3, 3, 7)])
@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 64, 16), ("float16", 33, 64), ("bfloat16", 72, 17), ("bfloat16", 128, 32),
                                              ("float16", 128, 128), ("float32", 32, 100), ("float32", 17, 16),
                                              ("float32", 64, 64), ("float32", 52, 33)])
@pytest.mark.parametrize("order", ["cell", "mixed"])
def test_edges_of_tiles_and_phases(gpu_handle, rows, ks, dtype_name, ci, co, order):
    import torch
    import mluop_hip as m
    print("dense, rows in LDS", rows, ks, dtype_name, ci, co, order, flush=True)
    rng = np.random.default_rng(rows + ci)
    idx = random_voxels(rng, 1, SPACE, rows, shuffle=order == "mixed")
    K = int(np.prod(ks))
    sub_m = all(k % 2 for k in ks)
    pad = [k // 2 for k in ks]
    out = [s + 2 * p - k + 1 for s, p, k in zip(SPACE, pad, ks)]
    pairs, _, num, n_out = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 1, SPACE, ks, out, pad,
                                              [1, 1, 1], [1, 1, 1], sub_m)
    counts = [int(v) for v in num.cpu()]
    pairs_np = pairs.cpu().numpy()
    feats = round_to(rng.uniform(-1, 1, (rows, ci)).astype(np.float32), dtype_name)
    dy = round_to(rng.uniform(-1, 1, (n_out, co)).astype(np.float32), dtype_name)
    b = 1.0 / np.sqrt(K * ci)
    w = round_to(rng.uniform(-b, b, (K, ci, co)).astype(np.float32), dtype_name)
    t_f, t_w, t_dy = (to_torch(a, dtype_name, "cuda") for a in (feats, w.reshape(tuple(ks) + (ci, co)), dy))
    gpu_handle.set_kernel_choice("dense_tiles", True)
    try:
        got = m.indice_conv_forward(gpu_handle, t_f, t_w, m.LAYOUT_ARRAY, pairs, counts, n_out, sub_m)
        dx = m.indice_conv_backward_data(gpu_handle, t_dy, t_w, m.LAYOUT_ARRAY, pairs, counts, sub_m, ci)
    finally:
        gpu_handle.set_kernel_choice("dense_tiles", None)
    check_close(from_torch(got), oracle.forward(feats, w, pairs_np, counts, n_out), dtype_name, "forward")
    check_close(from_torch(dx), oracle.backward_data(dy, w, pairs_np, counts), dtype_name, "backward_data")


# either side of the row counts up to which a phase has two pieces, and rows in no order, where it has two further on
@pytest.mark.parametrize("rows", [10000, 10001, 32768, 32769, 131072, 131073])
@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 64, 16), ("bfloat16", 128, 32), ("float16", 128, 64), ("bfloat16", 48, 64),
                                              ("float16", 64, 128)])
@pytest.mark.parametrize("order", ["cell", "mixed"])
def test_phases_of_one_and_two_pieces(gpu_handle, rows, dtype_name, ci, co, order):
    import torch
    import mluop_hip as m
    print("dense, pieces of a phase", rows, dtype_name, ci, co, order, flush=True)
    rng = np.random.default_rng(rows + ci)
    # (0.16 to 0.27 filled, uneven counts are summed by offset, in phases of one piece)
    space = (16 if 30000 < rows < 40000 else 8, 161, 163)
    cells = rng.choice(np.prod(space), rows, replace=False)
    cells = cells if order == "mixed" else np.sort(cells)
    idx = np.stack([0 * cells, cells // (161 * 163), cells // 163 % 161, cells % 163], 1).astype(np.int32)
    pairs, _, num, n_out = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 1, space, (3, 3, 3), space,
                                              [1, 1, 1], [1, 1, 1], [1, 1, 1], True)
    counts = [int(v) for v in num.cpu()]
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((rows, ci), generator=g, device="cuda").to(dtype)
    w = (torch.randn((27, ci, co), generator=g, device="cuda") * 0.1).to(dtype)
    gpu_handle.set_kernel_choice("dense_tiles", True)
    gpu_handle.set_kernel_timing(True)
    try:
        got = m.indice_conv_forward(gpu_handle, x, w.reshape(3, 3, 3, ci, co), m.LAYOUT_ARRAY, pairs, counts, n_out, True)
        torch.cuda.synchronize()
        names = [n for n, _ in gpu_handle.kernel_timings()]
        dx = m.indice_conv_backward_data(gpu_handle, got, w.reshape(3, 3, 3, ci, co), m.LAYOUT_ARRAY, pairs, counts,
                                         True, ci)
    finally:
        gpu_handle.set_kernel_timing(False)
        gpu_handle.set_kernel_choice("dense_tiles", None)
    assert "gatherConvDense" in names, names
    for result, source, forward in ((got, x, True), (dx, got, False)):
        want = torch.zeros(result.shape, dtype=torch.float64, device="cuda")
        size = torch.zeros_like(want)
        for k, n in enumerate(counts):
            i, j = pairs[k, 1 - forward, :n].long(), pairs[k, int(forward), :n].long()
            f = w[k].double() if forward else w[k].double().T
            want.index_add_(0, j, source[i].double() @ f)
            size.index_add_(0, j, source[i].double().abs() @ f.abs())
        # a chain of 27 products of `channels` terms, each step rounded once, and the result's own rounding
        rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dtype_name]
        bound = 27 * source.shape[1] * 2.0 ** -24 * size + rounding * want.abs() + 2.0 ** -25
        assert ((result.double() - want).abs() <= bound).all()
