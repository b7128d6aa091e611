"""Output cells of strided 3x3x3 and 2x2x2 rulebooks against a plain enumeration: candidates of a row that are
neighbours, that fall into two or three words of the bitmap, and rows in and out of order.  Axes with a stride have no
dilation: where that makes two cases alike, their clouds are two."""
import itertools

import numpy as np
import pytest

from spconv_cases import random_voxels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks", [3, 2])
@pytest.mark.parametrize("stride", [(2, 2, 2), (2, 2, 1), (1, 1, 2), (3, 1, 2), (2, 1, 1), (1, 2, 3)])
@pytest.mark.parametrize("dilation", [(1, 1, 1), (1, 1, 40), (2, 1, 65), (1, 3, 2)])
@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("rows", [1, 130, 1500])
def test_marked_cells(gpu_handle, ks, stride, dilation, shuffle, rows):
    import torch
    import mluop_hip as m
    print("strided marks", ks, stride, dilation, shuffle, rows, flush=True)
    cloud = [rows, ks, *stride, *dilation]
    dilation = tuple(d if s == 1 else 1 for d, s in zip(dilation, stride))  # (one of the two an axis)
    space, pad = (5, 7, 300), (1, 1, 1)
    idx = random_voxels(np.random.default_rng(cloud), 2, space, rows, shuffle=shuffle)
    ospace = [(n + 2 * p - d * (ks - 1) - 1) // s + 1 for n, p, s, d in zip(space, pad, stride, dilation)]
    if min(ospace) < 1:
        pytest.skip("no output space")
    pairs, rows_out, num, n_out = m.get_indice_pairs(gpu_handle, torch.from_numpy(idx).cuda(), 2, space, [ks] * 3,
                                                     ospace, list(pad), list(stride), list(dilation), False)
    torch.cuda.synchronize()
    lists, cells = [], set()
    for k in itertools.product(range(ks), repeat=3):
        at = idx[:, 1:].astype(np.int64) + np.array(pad) - np.array(k) * np.array(dilation)
        o = at // np.array(stride)
        ok = ((at >= 0) & (at % np.array(stride) == 0) & (o < np.array(ospace))).all(axis=1)
        lin = ((idx[:, 0] * ospace[0] + o[:, 0]) * ospace[1] + o[:, 1]) * ospace[2] + o[:, 2]
        lists.append((np.flatnonzero(ok), lin[ok]))
        cells.update(lin[ok].tolist())
    cells = np.array(sorted(cells), np.int64)
    assert n_out == len(cells)
    got = rows_out.cpu().numpy()[:n_out].astype(np.int64)
    assert (((got[:, 0] * ospace[0] + got[:, 1]) * ospace[1] + got[:, 2]) * ospace[2] + got[:, 3] == cells).all()
    pairs, num = pairs.cpu().numpy(), num.tolist()
    for k, (rows_in, lin) in enumerate(lists):
        assert num[k] == len(rows_in)
        assert (pairs[k, 0, :num[k]] == rows_in).all() and (cells[pairs[k, 1, :num[k]]] == lin).all()
