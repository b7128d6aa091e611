"""Tall tiles of 512 rows with two teams of multiplying waves (2-byte types, more than 32 offsets, rows of 33 channels
up): the bits of the pair-list kernel of short tiles at row counts around a tile, with offsets that fill whole
tiles, none and a few rows of them, and the fallback for lists that are not in order."""
import numpy as np
import pytest

from spconv_cases import check_close, from_torch
from test_gpu_tall_tiles import both_directions, check, make_case
import sparse_conv_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co", [(64, 64), (48, 100), (128, 128), (65, 65)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("rows,space", [(1, (4, 4, 4)), (511, (8, 9, 10)), (512, (8, 8, 8)), (513, (40, 60, 60)),
                                        (2049, (12, 20, 24))])
def test_bits_of_the_short_tiles(gpu_handle, ci, co, dtype_name, rows, space):
    print("tall teams", ci, co, dtype_name, rows, flush=True)
    check(gpu_handle, make_case(gpu_handle, rows, space, (3, 3, 5), ci, co, dtype_name, False), (True, True))


@pytest.mark.parametrize("foreign", [False, True])
def test_lists_that_are_not_in_order(gpu_handle, foreign):
    """Pairs written over after the library saw them in order, and pairs it has not seen: those are taken in order on
    trust, with the row map's kernels, whose tiles have another height, behind them."""
    import torch
    rows, space, ks, channels = 5000, (12, 24, 24), (3, 3, 5), 64  # (more than a grid rounded up to eight tiles covers)
    case = make_case(gpu_handle, rows, space, ks, channels, channels, "float16", False)
    pairs = case["pairs"].cpu().numpy().copy()
    rng = np.random.default_rng(3)
    for k, n in enumerate(case["num"]):
        order = rng.permutation(n)
        pairs[k, :, :n] = pairs[k][:, :n][:, order]
    if foreign:
        case["pairs"] = torch.from_numpy(pairs).cuda()
    else:
        case["pairs"].copy_(torch.from_numpy(pairs))
    out, dx, ran = both_directions(gpu_handle, case, True)
    torch.cuda.synchronize()
    assert ran == (True, True)
    w_k = from_torch(case["w"]).reshape(45, channels, channels)
    ref = oracle.forward(case["host"]["x"], w_k, pairs, case["num"], case["n_out"])
    check_close(from_torch(out), ref, "float16", "tall teams")
    ref = oracle.backward_data(case["host"]["dy"], w_k, pairs, case["num"])
    check_close(from_torch(dx), ref, "float16", "tall teams")
