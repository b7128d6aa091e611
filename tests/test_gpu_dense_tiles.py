"""The dense gather kernel's two tile shapes for rows above 128 bytes: which one runs goes by how full the number of
result rows leaves the last round of tiles (65 536 rows: wide from two thirds on), and both are held
to sums in 64 bits, on either side of the lines."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [219_999, 220_000, 220_129, 43_690, 43_691, 65_536, 65_537, 109_226, 109_227, 131_073,
                                  196_608, 196_609])
@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 128, 128), ("bfloat16", 96, 65), ("float32", 64, 100)])
@pytest.mark.parametrize("order", ["cell", "mixed"])
def test_forward_on_either_side_of_the_wide_tiles(gpu_handle, rows, dtype_name, ci, co, order):
    import torch
    import mluop_hip as m
    print("dense tiles", rows, dtype_name, ci, co, order, flush=True)
    if dtype_name == "float32" and rows == 220_000:
        rows = 220_001
    rng = np.random.default_rng(rows)
    space = (12, 170, 170)
    cells = rng.choice(space[0] * space[1] * space[2], rows, replace=False)
    if order == "cell":
        cells = np.sort(cells)
    idx = np.stack([np.zeros_like(cells), cells // (170 * 170), cells // 170 % 170, cells % 170], axis=1).astype(np.int32)
    pairs, _, num, n_out = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 1, space, (3, 3, 3), space,
                                              [1, 1, 1], [1, 1, 1], [1, 1, 1], True)
    counts = [int(v) for v in num.cpu()]
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((rows, ci), generator=g, device="cuda").to(dtype)
    w = (torch.rand((3, 3, 3, ci, co), generator=g, device="cuda") * 0.1 - 0.05).to(dtype)
    gpu_handle.set_kernel_choice("dense_tiles", True)
    try:
        got = m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, counts, n_out, True)
    finally:
        gpu_handle.set_kernel_choice("dense_tiles", None)
    ref = torch.zeros((rows, co), dtype=torch.float64, device="cuda")
    size = torch.zeros_like(ref)
    for k, n in enumerate(counts):
        i, o = pairs[k, 0, :n].long(), pairs[k, 1, :n].long()
        wk = w.reshape(27, ci, co)[k].double()
        ref.index_add_(0, o, x[i].double() @ wk)
        size.index_add_(0, o, x[i].double().abs() @ wk.abs())
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    # fp32 sums of 27 * ci products, one rounding to the type (halves below 2^-14 are spaced 2^-24 apart)
    bound = 2.0 ** -24 * 27 * ci * size + rounding * ref.abs() + (2.0 ** -25 if dtype_name == "float16" else 0)
    assert ((got.double() - ref).abs() <= bound).all()
    assert (got.double() - ref).norm() <= (2 * rounding + 1e-6) * ref.norm()
