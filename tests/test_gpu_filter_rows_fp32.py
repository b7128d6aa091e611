"""Backward filter, fp32 rows of more than 16 channels: the kernel whose rows go from memory to LDS as they are, against
the oracle and bit for bit against the kernel that stages them through registers (same products, same order of sums)."""
import pytest

import sparse_conv_oracle as oracle
from spconv_cases import check_close, from_torch, to_torch
from test_gpu_conv import conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    # (space, L, kernel, ci, co, sub_m, stride): slices of several chunks of row indices, ragged ends
    ((14, 20, 20), 4000, (3, 3, 3), 128, 128, True, (1, 1, 1)),
    ((14, 20, 20), 3100, (3, 3, 3), 64, 32, True, (1, 1, 1)),
    ((14, 20, 20), 3100, (3, 3, 3), 32, 32, True, (1, 1, 1)),
    ((12, 30, 30), 5000, (3, 3, 3), 32, 128, False, (2, 2, 2)),
    ((6, 6, 6), 150, (5, 5, 5), 64, 64, True, (1, 1, 1)),       # 125 offsets, short lists
    # rows that do not fill their blocks of channels: one block of two waves short, the last piece short, both
    ((14, 20, 20), 2500, (3, 3, 3), 48, 96, True, (1, 1, 1)),
    ((14, 20, 20), 2500, (3, 3, 3), 20, 68, True, (1, 1, 1)),
    ((12, 30, 30), 5000, (2, 2, 2), 112, 36, False, (2, 2, 2)),
    ((3, 4, 4), 3, (3, 3, 3), 32, 64, True, (1, 1, 1)),         # less than a multiply's pairs
])
def test_rows_in_lds_against_staging(gpu_handle, shape):
    import torch
    import mluop_hip
    space, L, ks, ci, co, sub_m, stride = shape
    print("backward filter case", shape, flush=True)
    c = conv_case(14, 1, space, L, ks, ci, co, sub_m, stride)
    feats = to_torch(c["feats"], "float32", "cuda")
    dy = to_torch(c["dy"], "float32", "cuda")
    pairs = torch.from_numpy(c["pairs"]).cuda()
    num_host = [int(v) for v in c["num"]]
    got = {}
    for staging in (False, True):
        gpu_handle.set_kernel_choice("filter_stores", True if staging else None)
        try:
            gpu_handle.set_kernel_timing(True)
            dw = mluop_hip.indice_conv_backward_filter(gpu_handle, feats, dy, pairs, num_host, c["ks"], sub_m)
            torch.cuda.synchronize()
            names = [k for k, _ in gpu_handle.kernel_timings()]
            gpu_handle.set_kernel_timing(False)
        finally:
            gpu_handle.set_kernel_choice("filter_stores", None)
        assert names[0] == ("backwardFilterMfma" if staging else "backwardFilterMfmaRows")
        got[staging] = dw
    ref = oracle.backward_filter(c["feats"], c["dy"], c["pairs"], c["num"], fast=True)
    check_close(from_torch(got[False]).reshape(ref.shape), ref, "float32", "backward_filter")
    assert torch.equal(got[False], got[True])
