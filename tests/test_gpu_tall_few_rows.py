"""Few result rows take the tall gather kernel's tiles of 128 rows: the bits of the pair-list kernel of short tiles in
both directions, at row counts around its tiles and at the last row count that is one tile a CU."""
import pytest

from test_gpu_pair_lists import kernels_of
from test_gpu_tall_tiles import make_case

pytestmark = pytest.mark.gpu


def both(handle, case, tall):
    import mluop_hip as m
    handle.set_kernel_choice("dense_tiles", False)
    handle.set_kernel_choice("tall_tiles", tall)
    try:
        out, forward = kernels_of(handle, lambda: m.indice_conv_forward(
            handle, case["x"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"], case["n_out"], case["sub_m"]))
        dx, backward = kernels_of(handle, lambda: m.indice_conv_backward_data(
            handle, case["dy"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"], case["sub_m"], case["ci"]))
    finally:
        handle.set_kernel_choice("dense_tiles", None)
        handle.set_kernel_choice("tall_tiles", None)
    return (out, dx) + tuple("gatherConvTall" in names or "gatherConvTall512" in names for names in (forward, backward))


def few(rows, q, c, size):
    q, c = (next(p for p in (16, 32, 64, 128) if p >= n) for n in (q, c))
    return c >= 64 and q * size <= 256 and rows >= 4096 and rows * (c // 64) <= 32768


@pytest.mark.parametrize("ci,co", [(64, 64), (5, 128), (16, 64), (33, 100), (64, 128)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("ks,rows,space", [((3, 3, 3), 4095, (9, 60, 100)), ((3, 3, 3), 4096, (9, 60, 100)),
                                           ((3, 3, 3), 4097, (9, 60, 100)), ((3, 3, 3), 4351, (9, 60, 100)),
                                           ((5, 5, 5), 4225, (9, 60, 100)), ((3, 3, 3), 16384, (20, 160, 160)),
                                           ((3, 3, 3), 16385, (20, 160, 160))])
def test_bits_of_the_short_tiles(gpu_handle, ci, co, dtype_name, ks, rows, space):
    import torch
    print("tall, few rows", ci, co, dtype_name, ks, rows, flush=True)
    case = make_case(gpu_handle, rows, space, ks, ci, co, dtype_name, False)
    out, dx, forward, backward = both(gpu_handle, case, None)
    ref_out, ref_dx, plain_f, plain_b = both(gpu_handle, case, False)
    torch.cuda.synchronize()
    assert torch.equal(out, ref_out) and torch.equal(dx, ref_dx) and not plain_f and not plain_b
    size = 4 if dtype_name == "float32" else 2
    assert forward == few(rows, ci, co, size) and backward == few(rows, co, ci, size)


@pytest.mark.parametrize("ci,co", [(64, 64), (16, 128), (128, 64)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("ks,rows,space", [((5, 5, 5), 1, (9, 60, 100)), ((5, 5, 5), 127, (9, 60, 100)),
                                           ((3, 3, 7), 128, (9, 60, 100)), ((5, 5, 5), 129, (9, 60, 100)),
                                           ((3, 3, 7), 1025, (9, 60, 100)), ((5, 5, 5), 4095, (9, 60, 100)),
                                           ((3, 1, 11), 2000, (9, 60, 100))])
def test_many_offsets_and_few_rows(gpu_handle, ci, co, dtype_name, ks, rows, space):
    import torch
    print("tall, few rows, many offsets", ci, co, dtype_name, ks, rows, flush=True)
    case = make_case(gpu_handle, rows, space, ks, ci, co, dtype_name, False)
    out, dx, forward, backward = both(gpu_handle, case, None)
    ref_out, ref_dx, _, _ = both(gpu_handle, case, False)
    torch.cuda.synchronize()
    assert torch.equal(out, ref_out) and torch.equal(dx, ref_dx)
    size = 4 if dtype_name == "float32" else 2
    assert forward == (ci * size <= 256) and backward == (co * size <= 256 and ci >= 64)


def test_no_step_between_few_rows_and_more(gpu_handle):
    """125 offsets, fp32: in tiles of 256 rows 4095 rows took 1.4 times as long as 4097 rows in tiles of 128."""
    import mluop_hip as m
    times = []
    for rows in (4095, 4097):
        case = make_case(gpu_handle, rows, (9, 60, 100), (5, 5, 5), 64, 64, "float32", False)
        runs = []
        for _ in range(12):
            gpu_handle.set_kernel_timing(True)
            try:
                m.indice_conv_forward(gpu_handle, case["x"], case["w"], m.LAYOUT_ARRAY, case["pairs"], case["num"],
                                      case["n_out"], case["sub_m"])
                runs += [ms for name, ms in gpu_handle.kernel_timings() if name == "gatherConvTall"]
            finally:
                gpu_handle.set_kernel_timing(False)
        times.append(sorted(runs)[len(runs) // 2])
    print("125 offsets, 4095 and 4097 rows: %.1f, %.1f us" % (times[0] * 1e3, times[1] * 1e3), flush=True)
    assert times[0] < 1.2 * times[1]
