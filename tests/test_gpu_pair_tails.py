"""mluOpExtSetPairTails: without the -1 behind each offset's pairs the lists, counts and output rows are the same,
for every probe kernel and both row orders, and the next rulebook has its -1 again."""
import numpy as np
import pytest

from spconv_cases import out_space, random_voxels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks,stride,dilation,sub_m", [((3, 3, 3), 1, 1, True), ((5, 5, 5), 1, 1, True), ((3, 1, 7), 1, 1, True),
                                                      ((3, 3, 3), 1, 2, False), ((3, 3, 3), 2, 1, False),
                                                      ((2, 2, 2), 2, 1, False), ((3, 3, 1), 2, 1, False),
                                                      ((3, 3, 3), 1, 1, False)])
@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("rows", [1, 64, 1300])
def test_lists_without_tails(gpu_handle, ks, stride, dilation, sub_m, shuffle, rows):
    import torch
    import mluop_hip as m
    print("pair tails", ks, stride, dilation, sub_m, shuffle, rows, flush=True)
    space = (9, 18, 20)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(rows), 1, space, rows, shuffle=shuffle)).cuda()
    pad = [dilation * (k // 2) for k in ks]
    dil = [dilation] * 3
    ospace = list(space) if sub_m else out_space(space, ks, pad, [stride] * 3, dil)

    def build(**kwargs):
        return m.get_indice_pairs(gpu_handle, idx, 1, space, ks, ospace, pad, [stride] * 3, dil, sub_m, **kwargs)

    pairs, rows_out, num, n_out = build()
    bare, bare_rows, bare_num, bare_n = build(tails=False)
    again = build()
    assert torch.equal(num, bare_num) and n_out == bare_n and torch.equal(rows_out, bare_rows)
    for k, n in enumerate(num.cpu().tolist()):
        assert torch.equal(pairs[k, :, :n], bare[k, :, :n])
        assert (pairs[k, :, n:] == -1).all() and torch.equal(pairs[k], again[0][k])
