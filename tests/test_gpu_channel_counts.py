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


@pytest.mark.parametrize("rows", [1, 2, 3])
@pytest.mark.parametrize("channels,dtype_name", [(65, "float16"), (80, "float16"), (95, "bfloat16"), (127, "bfloat16"),
                                                 (33, "float32"), (47, "float32"), (64, "float32")])
def test_a_tensor_shorter_than_the_last_chunk_of_a_row(gpu_handle, rows, channels, dtype_name):
    """Rows above 128 bytes go through the dense kernel in 64-byte chunks, and a tensor of one short
    row ends in front of the last of them: what lies behind it reads as zeros, in both directions."""
    print("short tensor", rows, channels, dtype_name, flush=True)
    c = conv_case(rows + channels, 1, (4, 4, 4), rows, (3, 3, 3), channels, channels, True)
    gpu_handle.set_kernel_choice("dense_tiles", True)
    try:
        run_all_ops(gpu_handle, c, dtype_name, check=("fwd", "bwd_data"))
    finally:
        gpu_handle.set_kernel_choice("dense_tiles", None)
