"""Channel counts between the matrix-core tiles (rows that end inside a 16-byte piece, inside a
chunk, inside a column block), at row counts around the ends of a tile, for the tile-compacting and
the register-accumulating kernels."""

import pytest

from test_gpu_conv import conv_case, run_all_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co", [(1, 1), (4, 16), (5, 17), (12, 33), (24, 48), (48, 24), (65, 96), (96, 127), (127, 5)])
@pytest.mark.parametrize("rows,dense", [(127, 1), (129, 0), (256, 1), (257, 1), (511, 0), (513, 1)])
@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
def test_any_channel_count_matches_oracle(gpu_handle, ci, co, rows, dense, dtype_name):
    print("channels", ci, co, "rows", rows, "dense", dense, dtype_name, flush=True)
    c = conv_case(rows + ci, 1, (8, 9, 10), rows, (3, 3, 3), ci, co, True)
    gpu_handle.set_kernel_choice("dense_tiles", bool(dense))
    try:
        run_all_ops(gpu_handle, c, dtype_name)
    finally:
        gpu_handle.set_kernel_choice("dense_tiles", None)
