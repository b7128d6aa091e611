"""Backward filter of a layer whose output gradient has 2 to 4 GiB (a million strewn voxels reach 27 million cells): the kernel
that addresses rows with 32-bit byte offsets, up to the last row it can reach and the kernel beyond it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L, KS = 1_000_000, (3, 3, 3)
GIB2 = 1 << 31


@pytest.mark.parametrize("dtype_name,ci,co,rows,kernel", [
    ("float16", 64, 64, GIB2 // 128 - 1, "backwardFilterMfmaTr"),
    ("float16", 64, 64, GIB2 // 128 + 70_000, "backwardFilterMfmaTr"),
    ("bfloat16", 48, 56, GIB2 // 112 + 70_000, "backwardFilterMfmaTr"),       # rows that do not fill their blocks
    ("bfloat16", 32, 128, 0xfffffe00 // 256, "backwardFilterMfmaTr"),         # the last byte there can be
    ("float16", 32, 80, 0xfffffe00 // 160, "backwardFilterMfmaTr"),
    ("float16", 32, 128, 0xfffffe00 // 256 + 1, "backwardFilterMfma"),        # (and the last row of the API's tensors)
    ("float32", 32, 32, GIB2 // 128 + 70_000, "backwardFilterMfmaRows"),
    ("float32", 20, 40, 0xfffffe00 // 160 - 3, "backwardFilterMfmaRows"),
    ("float32", 32, 64, 0xfffffe00 // 256 + 1, "backwardFilterMfma"),
])
def test_output_gradients_of_more_than_2_gib(gpu_handle, dtype_name, ci, co, rows, kernel):
    import torch
    import mluop_hip as m
    print("long output gradient", dtype_name, ci, co, rows, flush=True)
    dtype = getattr(torch, dtype_name)
    counts = [0] * 27
    counts[0], counts[5], counts[13], counts[26] = 3000, 1, 700, 64
    g = torch.Generator(device="cuda").manual_seed(ci)
    rng = np.random.default_rng(co)
    pairs = torch.full((27, 2, L), -1, dtype=torch.int32, device="cuda")
    x = torch.randn((L, ci), generator=g, device="cuda").to(dtype)
    dy = torch.zeros((rows, co), dtype=dtype, device="cuda")
    want = torch.zeros((27, ci, co), dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    for k, n in enumerate(counts):
        if n == 0:
            continue
        i = np.sort(rng.choice(L, n, replace=False))
        o = np.sort(rng.choice(rows, n, replace=False))
        i[-1], o[-1] = L - 1, rows - 1
        o[0] = min(o[0], GIB2 // (co * dy.element_size()) - 1)
        i, o = torch.from_numpy(i).cuda(), torch.from_numpy(o).cuda()
        dy[o] = torch.randn((n, co), generator=g, device="cuda").to(dtype)
        pairs[k, 0, :n], pairs[k, 1, :n] = i.int(), o.int()
        if n > 100:   # (pairs that name no row add nothing: the kernels look at every index)
            pairs[k, 0, 7], pairs[k, 1, 9], pairs[k, 1, 50] = -1, rows, -5
    for k, n in enumerate(counts):
        keep = [p for p in range(n) if n <= 100 or p not in (7, 9, 50)]
        i, o = (pairs[k, c, :n][keep].long() for c in (0, 1))
        a, b = x[i].double(), dy[o].double()
        want[k] = a.T @ b
        size[k] = a.abs().T @ b.abs()
    gpu_handle.set_kernel_timing(True)
    dw = m.indice_conv_backward_filter(gpu_handle, x, dy, pairs, counts, KS, False)
    torch.cuda.synchronize()
    names = [name for name, _ in gpu_handle.kernel_timings()]
    gpu_handle.set_kernel_timing(False)
    assert names[0] == kernel, names
    # sums of up to 3000 products in fp32, each step's rounding bounded by the sum of sizes; then one rounding
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    bound = 3000 * 2.0 ** -24 * size + rounding * want.abs() + 2.0 ** -25
    assert ((dw.reshape(27, ci, co).double() - want).abs() <= bound).all()
