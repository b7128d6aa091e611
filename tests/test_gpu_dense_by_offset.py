"""Layers whose pairs are too few for the register-accumulating kernel's one chain of sums a row, and many enough for the
same kernel with each offset's product by itself (2-byte types, 33 channels up on both sides): the pair-list kernels'
bits, for whole rows and rows that do not fill their fragments, and for a filter that is not finite."""
import numpy as np
import pytest

from spconv_cases import round_to, to_torch
from test_gpu_pair_lists import gpu_rulebook, kernels_of
from test_gpu_tall_teams import with_and_without_a_wait

pytestmark = pytest.mark.gpu


def floors_and_walls(space, fill, seed):
    """Cells of sheets two cells thick, `fill` of them present, in the order of their cells."""
    d, h, w = space
    z, y, x = np.meshgrid(np.arange(d), np.arange(h), np.arange(w), indexing="ij")
    there = (z // 2 % 4 == 0) | (y // 2 % 12 == 3)
    there &= np.random.default_rng(seed).random(there.shape) < fill
    cells = np.argwhere(there)
    return np.ascontiguousarray(np.concatenate([np.zeros((len(cells), 1)), cells], axis=1).astype(np.int32))


SMALL, LARGE = (17, 40, 44), (25, 160, 160)


@pytest.mark.parametrize("ci,co,space", [(64, 64, SMALL), (48, 40, SMALL), (128, 64, SMALL), (120, 56, SMALL),
                                         (64, 128, LARGE), (128, 128, LARGE), (72, 104, LARGE)])
@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("finite", [True, False])
def test_bits_of_the_pair_list_kernels(gpu_handle, ci, co, space, dtype_name, finite):
    import torch
    import mluop_hip as m
    print("dense by offset", ci, co, space, dtype_name, finite, flush=True)
    idx = floors_and_walls(space, 0.37, ci + co)
    ks = (3, 3, 3)
    pairs, num, n_out = gpu_rulebook(gpu_handle, idx, 1, space, ks, [1, 1, 1], [2, 2, 2], [1, 1, 1], False)
    fill = sum(num) / n_out / 27
    rest = sorted(num)
    assert 0.16 <= fill < 0.27 and 1.1 <= rest[-2] / (sum(rest[:-1]) / 26) < 1.5 and (co <= 64 or n_out >= 30000), (fill, n_out)
    rng = np.random.default_rng(ci)
    x = to_torch(round_to(rng.standard_normal((idx.shape[0], ci)).astype(np.float32), dtype_name), dtype_name, "cuda")
    w = to_torch(round_to((rng.standard_normal(ks + (ci, co)) / np.sqrt(27 * ci)).astype(np.float32), dtype_name), dtype_name, "cuda")
    if not finite:
        w[0, 1, 2, 3, 4] = float("inf")
    got = {}
    for lists in (False, True):
        gpu_handle.set_kernel_choice("dense_tiles", False if lists else None)
        try:
            got[lists], names = kernels_of(gpu_handle, lambda: m.indice_conv_forward(
                gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, num, n_out, False))
        finally:
            gpu_handle.set_kernel_choice("dense_tiles", None)
        assert ("gatherConvDenseByOffset" in names) != lists and "gatherConvDense" not in names, names
    a, b = got[False], got[True]
    if finite:
        assert torch.equal(a, b)
    else:  # (an offset whose filter is not finite goes first: the others' sums of its column only)
        keep = torch.ones(co, dtype=torch.bool)
        keep[4] = False
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)) and not bool(torch.isfinite(a).all())
        error = (a.double() - b.double())[:, keep].abs().max()
        assert float(error) <= 2.0 ** (-7 if dtype_name == "bfloat16" else -10) * float(b[:, keep].double().abs().max())


def test_row_map_behind_lists_on_trust():
    """Rows out of order: the row map's kernel adds in the same order, whether the host knew or launched on trust."""
    import torch
    import mluop_hip as m
    ks, channels, space = (3, 3, 3), 64, (24, 24, 24)
    idx = floors_and_walls(space, 0.3, 5)  # (a submanifold layer: a strided one's rulebook waits for its rows)
    rng = np.random.default_rng(6)
    idx = np.ascontiguousarray(idx[rng.permutation(len(idx))])
    x = torch.from_numpy(rng.standard_normal((idx.shape[0], channels)).astype(np.float32)).cuda().half()
    w = torch.from_numpy((rng.standard_normal(ks + (channels, channels)) / 40).astype(np.float32)).cuda().half()
    ((want, known), (got, trusted)), fill = with_and_without_a_wait(m.make_handle_on_current_stream(), idx, space, ks, 1, x, w)
    assert 0.16 <= fill < 0.27, fill
    dense = {"gatherConvDense", "gatherConvDenseByOffset"}
    assert "packFilterCutPairLists" not in known and not dense & set(known), known
    assert "packFilterCutPairLists" in trusted and [n for n in trusted if n in dense] == ["gatherConvDenseByOffset"], trusted
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,density", [(300, 0.18), (700, 0.25), (1500, 0.2), (6000, 0.2)])
@pytest.mark.parametrize("ks", [(3, 3, 3), (5, 5, 5)])
def test_strewn_voxels_stay_with_the_pair_lists(gpu_handle, rows, density, ks):
    """Their counts differ by chance, by a tenth of the mean and more at few rows; and 125 offsets, whatever they differ by."""
    import torch
    import mluop_hip as m
    rng = np.random.default_rng(rows)
    side = int(round((rows / density) ** (1 / 3)))
    cells = np.sort(rng.choice(side ** 3, rows, replace=False))
    idx = np.stack([0 * cells, cells // side ** 2, cells // side % side, cells % side], 1).astype(np.int32)
    pairs, num, n_out = gpu_rulebook(gpu_handle, idx, 1, (side,) * 3, ks, [k // 2 for k in ks], [1, 1, 1], [1, 1, 1], True)
    x = torch.randn((rows, 64), device="cuda").half()
    w = torch.randn(ks + (64, 64), device="cuda").half()
    _, names = kernels_of(gpu_handle, lambda: m.indice_conv_forward(gpu_handle, x, w, m.LAYOUT_ARRAY, pairs, num, n_out, True))
    assert not any(n.startswith("gatherConvDense") for n in names), names
