"""Submanifold rulebooks of few rows, which one launch builds, against those of the launches for larger ones: the same
pairs, counts, rows, tails and report, for rows in and out of order, cells named twice and rows outside the space."""
import numpy as np
import pytest

from spconv_cases import random_voxels
from test_gpu_pair_lists import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks,dilation,pad", [((3, 3, 3), 1, None), ((5, 5, 5), 1, None), ((3, 1, 7), 2, None), ((1, 1, 1), 1, None),
                                             ((2, 3, 4), 1, (1, 0, 2)), ((3, 3, 3), 1, (0, 1, 2))])
@pytest.mark.parametrize("order", ["cell", "mixed", "twice", "outside"])
@pytest.mark.parametrize("rows", [1, 63, 1024, 1025, 3001, 4096, 4097])
def test_pairs_of_the_general_launches(gpu_handle, ks, dilation, pad, order, rows):
    import torch
    import mluop_hip as m
    print("small rulebook", ks, dilation, pad, order, rows, flush=True)
    rng = np.random.default_rng(rows)
    space = (9, 24, 20)
    idx = random_voxels(rng, 2, space, rows, shuffle=order != "cell")
    if order == "twice":
        idx[rows // 2:] = idx[:rows - rows // 2]
    elif order == "outside":
        some = rng.integers(0, rows, rows // 3 + 1)
        idx[some, rng.integers(0, 4, some.size)] = rng.choice([-1, -3, 2, 9, 10, 24, 25, 100], some.size)
    idx = torch.from_numpy(np.ascontiguousarray(idx)).cuda()
    dil = [dilation] * 3
    pad = [dilation * (k // 2) for k in ks] if pad is None else list(pad)

    def build(small, tails):
        gpu_handle.set_kernel_choice("small_rulebook", small)
        try:
            return kernels_of(gpu_handle, lambda: m.get_indice_pairs(gpu_handle, idx, 2, space, ks, list(space), pad,
                                                                     [1] * 3, dil, True, out_rows=rows + 5, tails=tails))
        finally:
            gpu_handle.set_kernel_choice("small_rulebook", None)

    try:
        (ref, ref_rows, ref_num, n_ref), ran = build(False, True)
    except m.MluOpError as refused:
        with pytest.raises(m.MluOpError) as again:
            build(None, True)
        assert str(again.value) == str(refused)
        return
    assert "rbSubmSmall" not in ran
    for tails in (True, False):
        (pairs, rows_out, num, n), ran = build(None, tails)
        assert ("rbSubmSmall" in ran) == (rows <= 4096)
        assert torch.equal(num, ref_num) and n == n_ref and torch.equal(rows_out, ref_rows)
        for k, count in enumerate(num.tolist()):
            assert torch.equal(pairs[k, :, :count], ref[k, :, :count])
            assert not tails or torch.equal(pairs[k], ref[k])
