"""A SparseSequential waits for its rulebooks' pair counts once, behind the last of them: also for more rulebooks than
a handle keeps counts of, and when building one of them fails."""
import numpy as np
import pytest

from spconv_cases import random_voxels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rulebooks,rows", [(1, 1), (3, 500), (40, 300)])
def test_counts_of_every_rulebook(gpu_handle, rulebooks, rows):
    import torch
    from mluop_hip import get_indice_pairs, nn as spnn
    print("pending counts", rulebooks, rows, flush=True)
    space = (9, 20, 20)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(rows), 1, space, rows)).cuda()
    net = spnn.SparseSequential(*[spnn.SubMConv3d(4, 4, 3, dilation=1) for _ in range(rulebooks - 1)],
                                spnn.SparseConv3d(4, 4, 3, stride=2, padding=1)).cuda()
    t = spnn.SparseTensor(torch.randn(rows, 4, device="cuda"), idx, space, 1, distinct=True)
    net.plan(t)
    assert len(t.rulebooks) == rulebooks
    for rb in t.rulebooks.values():
        assert isinstance(rb._indice_num, list)
        pad, stride = ([1] * 3, [1] * 3) if rb.sub_m else ([1] * 3, [2] * 3)
        _, _, num, n_out = get_indice_pairs(gpu_handle, idx, 1, space, (3, 3, 3), rb.out_space, pad, stride, [1] * 3, rb.sub_m)
        assert rb.indice_num == num.tolist() and rb.num_act_out == n_out


def test_counts_behind_a_layer_that_fails(gpu_handle):
    import torch
    from mluop_hip import nn as spnn
    space = (9, 20, 20)
    idx = torch.from_numpy(random_voxels(np.random.default_rng(2), 1, space, 200)).cuda()
    net = spnn.SparseSequential(spnn.SubMConv3d(4, 4, 3), spnn.SparseInverseConv3d(4, 4, 3, indice_key="none")).cuda()
    t = spnn.SparseTensor(torch.randn(200, 4, device="cuda"), idx, space, 1, distinct=True)
    with pytest.raises(AssertionError):
        net(t)
    (rb,) = t.rulebooks.values()
    assert isinstance(rb._indice_num, list) and sum(rb.indice_num) > 0
