"""Output rows of a regular rulebook are the marked cells in ascending order, whatever share of a word's, a wavefront's
or a block's cells is marked, and however many workgroups take the cells of a block of 256 words (16384 cells)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,rest", [(0, 1), (0, 63), (1, 0), (1, 1), (3, 77), (191, 0), (192, 5), (513, 1), (1535, 9),
                                         (1536, 0), (1537, 64), (4097, 3)])
@pytest.mark.parametrize("marks", ["all", "runs", "few"])
def test_rows_are_the_cells_in_order(gpu_handle, blocks, rest, marks):
    import torch
    import mluop_hip as m
    print("decode cells", blocks, rest, marks, flush=True)
    n = blocks * 16384 + rest
    rng = np.random.default_rng(blocks + rest)
    if marks == "all":
        cells = np.arange(n) if n < 200000 else np.concatenate([np.arange(70000), np.arange(n - 70000, n)])
    elif marks == "runs":  # full words, words of one cell, empty ones
        cells = np.unique(np.concatenate([np.arange(s, min(s + l, n)) for s, l in
                                          zip(rng.integers(0, n, 64), rng.integers(1, 700, 64))]))
    else:
        cells = np.unique(rng.integers(0, n, 3000))
    cells = np.union1d(cells, [0, n - 1])
    # a grid one cell wide keeps the cell's number as a coordinate; rows in no order
    indices = np.zeros((cells.size, 4), np.int32)
    indices[:, 1] = rng.permutation(cells)
    pairs, rows, num, n_out = m.get_indice_pairs(gpu_handle, torch.from_numpy(indices).cuda(), 1, (n, 1, 1), (1, 1, 1),
                                                 (n, 1, 1), [0] * 3, [1] * 3, [1] * 3, False)
    torch.cuda.synchronize()
    assert n_out == cells.size
    got = rows.cpu().numpy()[:n_out]
    assert (got[:, 1] == cells).all() and (got[:, [0, 2, 3]] == 0).all()
    pairs = pairs.cpu().numpy()[0, :, :n_out]
    assert (indices[pairs[0], 1] == cells[pairs[1]]).all()
