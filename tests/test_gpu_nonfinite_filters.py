"""A filter with an infinity or a NaN in the slice of one offset: it reaches the result rows that have
a pair at that offset, and no other row, whichever kernel the pair counts select.  (The kernels that
multiply whole tiles of rows would otherwise spread it: zero times infinity is a NaN.)"""
import numpy as np
import pytest

import sparse_conv_oracle as oracle
from spconv_cases import check_close, from_torch, random_voxels, round_to, to_torch

pytestmark = pytest.mark.gpu

KERNELS = {
    "dense": ({"dense_tiles": True}, "gatherConvDense"),
    "pairs": ({"dense_tiles": False, "wave_per_tile": False}, "gatherConvMfma"),
    "wave": ({"dense_tiles": False}, "gatherConvWave"),
    "simt": ({"gather_simt": True}, "gatherConvSimt"),
}


def check_rows(got, ref, dtype_name, what):
    """The same elements are finite, and those agree."""
    assert np.array_equal(np.isfinite(got), np.isfinite(ref)), "%s: %d elements are not finite, the reference has %d" % (
        what, (~np.isfinite(got)).sum(), (~np.isfinite(ref)).sum())
    keep = np.isfinite(ref)
    if keep.any():
        check_close(got[keep], ref[keep], dtype_name, what)


def run(handle, kernel, dtype_name, ci, co, rows, space, order, offset, value, ks=(3, 3, 3)):
    import torch
    import mluop_hip as m
    rng = np.random.default_rng(rows + ci + offset)
    idx = random_voxels(rng, 1, space, rows, shuffle=order == "mixed")
    K = int(np.prod(ks))
    pairs, _, num, n_out = m.get_indice_pairs(handle, torch.from_numpy(idx).cuda(), 1, space, ks, space,
                                              [k // 2 for k in ks], [1, 1, 1], [1, 1, 1], True)
    num_host = [int(v) for v in num.cpu()]
    pairs_np = pairs.cpu().numpy()
    feats = round_to(rng.uniform(0.5, 1.5, (rows, ci)).astype(np.float32), dtype_name)
    dy = round_to(rng.uniform(0.5, 1.5, (rows, co)).astype(np.float32), dtype_name)
    b = 1.0 / np.sqrt(K * ci)
    w = round_to(rng.uniform(-b, b, (K, ci, co)).astype(np.float32), dtype_name)
    w[offset, ci // 2, co // 2] = value
    t_f, t_w, t_dy = (to_torch(a, dtype_name, "cuda") for a in (feats, w.reshape(tuple(ks) + (ci, co)), dy))
    choices, name = KERNELS[kernel]
    for which, on in choices.items():
        handle.set_kernel_choice(which, on)
    try:
        handle.set_kernel_timing(True)
        out = m.indice_conv_forward(handle, t_f, t_w, m.LAYOUT_ARRAY, pairs, num_host, n_out, True)
        dx = m.indice_conv_backward_data(handle, t_dy, t_w, m.LAYOUT_ARRAY, pairs, num_host, True, ci)
        names = [n for n, _ in handle.kernel_timings()]
    finally:
        handle.set_kernel_timing(False)
        for which in choices:
            handle.set_kernel_choice(which, None)
    assert name in names, names
    check_rows(from_torch(out), oracle.forward(feats, w, pairs_np, num_host, n_out), dtype_name, "forward")
    check_rows(from_torch(dx), oracle.backward_data(dy, w, pairs_np, num_host), dtype_name, "backward_data")


# (rows, space): most slots filled, few filled, and hardly any (tiles without a pair at most offsets,
# so that the number of offsets a tile walks is odd and even)
CLOUDS = [(300, (8, 9, 10)), (513, (20, 20, 20)), (40, (12, 12, 12)), (41, (12, 12, 12))]


@pytest.mark.parametrize("kernel", ["dense", "pairs"])
@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 16, 16), ("bfloat16", 64, 64), ("float16", 128, 128),
                                              ("bfloat16", 48, 24), ("float32", 16, 32), ("float32", 32, 16),
                                              ("float32", 64, 64), ("float16", 64, 128)])
@pytest.mark.parametrize("rows,space", CLOUDS)
@pytest.mark.parametrize("order", ["cell", "mixed"])
def test_matrix_core_kernels(gpu_handle, kernel, dtype_name, ci, co, rows, space, order):
    print("non-finite filter", kernel, dtype_name, ci, co, rows, order, flush=True)
    for offset, value in ((0, np.inf), (4, -np.inf), (26, np.nan)):
        run(gpu_handle, kernel, dtype_name, ci, co, rows, space, order, offset, value)


def test_wave_kernel(gpu_handle):
    for rows, space in CLOUDS:
        run(gpu_handle, "wave", "float16", 32, 32, rows, space, "cell", 0, np.inf)


@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
def test_generic_kernel(gpu_handle, dtype_name):
    for rows, space in CLOUDS:
        for ci, co in ((5, 70), (33, 130)):
            run(gpu_handle, "simt", dtype_name, ci, co, rows, space, "mixed", 0, np.inf)


@pytest.mark.parametrize("kernel", ["dense", "pairs"])
def test_a_filter_slice_in_a_later_chunk_of_offsets(gpu_handle, kernel):
    """125 offsets: the kernels take them in chunks of 27 or 28."""
    for dtype_name, c in (("float16", 32), ("float16", 64), ("bfloat16", 128)):
        for offset in (30, 81, 124):
            run(gpu_handle, kernel, dtype_name, c, c, 300, (8, 9, 10), "cell", offset, np.inf, ks=(5, 5, 5))
