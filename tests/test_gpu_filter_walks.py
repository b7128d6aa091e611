"""Backward filter by walks (many pairs): every pair of every offset is multiplied once, whatever the lengths of
the lists are, on both kernels, for types and channel counts on either side of a step, and with offsets that
have fewer pairs than a share has workgroups, or none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lists(rng, rows, counts):
    """[K, 2, rows] pair lists of the given lengths: distinct rows in ascending order on both sides."""
    pairs = np.full((len(counts), 2, rows), -1, dtype=np.int32)
    for k, n in enumerate(counts):
        for side in range(2):
            pairs[k, side, :n] = np.sort(rng.choice(rows, n, replace=False))
    return pairs


@pytest.mark.parametrize("dtype_name,ci,co", [("float16", 128, 128), ("bfloat16", 96, 100), ("float16", 64, 128),
                                              ("bfloat16", 32, 64), ("float16", 16, 16), ("float32", 32, 32)])
@pytest.mark.parametrize("spread", ["even", "uneven"])
def test_every_pair_counts_once(gpu_handle, dtype_name, ci, co, spread):
    import torch
    import mluop_hip as m
    print("filter walks", dtype_name, ci, co, spread, flush=True)
    rng = np.random.default_rng(ci + co)
    rows = 70_001
    if spread == "even":
        counts = [60_000 + int(v) for v in rng.integers(0, 9_999, 27)]
    else:  # (submanifold layers have their longest list in the middle)
        counts = [0, 1, 7, 63, 64, 65, 255, 256, 257, 2047, 2049, 69_999, 70_000, 70_001, 70_000, 69_998, 35_000, 12_345,
                  69_000, 68_000, 66_666, 51_200, 70_000, 69_000, 68_888, 70_001, 61_441]
    assert sum(counts) > 800_000
    pairs = torch.from_numpy(lists(rng, rows, counts)).cuda()
    dtype = getattr(torch, dtype_name)
    g = torch.Generator(device="cuda").manual_seed(ci)
    x = torch.randn((rows, ci), generator=g, device="cuda").to(dtype)
    dy = (torch.randn((rows, co), generator=g, device="cuda") * 0.1).to(dtype)
    got = m.indice_conv_backward_filter(gpu_handle, x, dy, pairs, counts, (3, 3, 3), False)
    again = m.indice_conv_backward_filter(gpu_handle, x, dy, pairs, counts, (3, 3, 3), False)
    torch.cuda.synchronize()
    assert torch.equal(got, again)
    got = got.reshape(27, ci, co).double()
    rounding = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8, "float32": 2.0 ** -24}[dtype_name]
    for k, n in enumerate(counts):
        a, b = x[pairs[k, 0, :n].long()].double(), dy[pairs[k, 1, :n].long()].double()
        ref, size = a.t() @ b, a.abs().t() @ b.abs()
        # fp32 sums: a walk adds at most an eighth of the offset's pairs, and no more than 64 tiles follow one
        # another in the sum; then one rounding to the type (halves below 2^-14 are spaced 2^-24 apart)
        bound = 2.0 ** -24 * (max(n, 1) / 8 + 64) * size + rounding * ref.abs() + (2.0 ** -25 if dtype_name == "float16" else 0)
        worst = ((got[k] - ref).abs() - bound).max().item() if n else got[k].abs().max().item()
        assert worst <= 0, (k, n, worst)
        # a pair that is missing or counted twice stands out among the sums of this offset
        if n >= 64:
            assert (got[k] - ref).norm() <= 1e-5 * size.norm() + 2 * rounding * ref.norm()
