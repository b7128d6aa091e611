"""Mean of the voxels' points by the library's kernel (mean_voxel_features without a gradient): against float64, at
vectors of four features and single ones, points around the four running sums, unaligned rows and voxels without a
point; and the calls that stay with torch."""
import pytest

pytestmark = pytest.mark.gpu


def launched(monkeypatch, call):
    """(the call's result, whether the library's kernel made it)"""
    import mluop_hip
    from mluop_hip import nn as spnn
    real, calls = mluop_hip.native(), []

    class Watched:
        def __getattr__(self, name):
            if name == "mean_voxel_points":
                calls.append(name)
            return getattr(real, name)
    with monkeypatch.context() as m:
        m.setattr(spnn, "native", lambda: Watched())
        return call(), bool(calls)


@pytest.mark.parametrize("features", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("points", [1, 3, 4, 5, 7, 32])
@pytest.mark.parametrize("voxels,skew", [(1, 0), (64, 0), (257, 1), (5000, 0)])
def test_against_float64(monkeypatch, features, points, voxels, skew):
    import torch
    from mluop_hip import nn as spnn
    print("mean", features, points, voxels, skew, flush=True)
    g = torch.Generator(device="cuda").manual_seed(voxels + points)
    flat = torch.randn(voxels * points * features + skew, device="cuda", generator=g)
    x = flat[skew:].view(voxels, points, features)
    counts = torch.randint(0, points + 1, (voxels,), device="cuda", generator=g, dtype=torch.int32)
    got, native = launched(monkeypatch, lambda: spnn.mean_voxel_features(x, counts))
    assert native
    by = counts.clamp(min=1).double().unsqueeze(1)
    ref = x.double().sum(dim=1) / by
    # every one of at most `points` additions and the division rounds once
    bound = (points + 1) * 2.0 ** -24 * x.double().abs().sum(dim=1) / by
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("points", [127, 128, 129, 4000])
def test_many_points_a_voxel_stay_with_torch(monkeypatch, points):
    """(whose reduction takes them side by side: 30 voxels of 4000 points in 35 us, one after the other in 635)"""
    import torch
    from mluop_hip import nn as spnn
    x = torch.randn(30, points, 16, device="cuda")
    counts = torch.full((30,), points, device="cuda", dtype=torch.int32)
    got, native = launched(monkeypatch, lambda: spnn.mean_voxel_features(x, counts))
    assert native == (points <= 128)
    bound = (points + 1) * 2.0 ** -24 * x.double().abs().mean(dim=1)
    assert bool(((got.double() - x.double().mean(dim=1)).abs() <= bound).all())


def test_what_stays_with_torch(monkeypatch):
    import torch
    from mluop_hip import nn as spnn
    x = torch.randn(50, 5, 4, device="cuda")
    counts = torch.randint(1, 6, (50,), device="cuda", dtype=torch.int32)
    ref = x.double().sum(dim=1) / counts.double().unsqueeze(1)
    leaf = x.clone().requires_grad_()
    out, native = launched(monkeypatch, lambda: spnn.mean_voxel_features(leaf, counts))
    assert not native
    (grad,) = torch.autograd.grad(out, leaf, torch.ones_like(out))
    assert torch.allclose(grad, (1.0 / counts.float())[:, None, None].expand_as(x))
    with torch.no_grad():
        assert launched(monkeypatch, lambda: spnn.mean_voxel_features(leaf, counts))[1]
    for voxels, n in ((x.half(), counts), (x.double(), counts), (x, counts.long()), (x[:0], counts[:0]),
                      (x.transpose(0, 1).contiguous().transpose(0, 1), counts), (x.cpu(), counts.cpu())):
        out, native = launched(monkeypatch, lambda: spnn.mean_voxel_features(voxels, n))
        assert not native and out.dtype == voxels.dtype and out.shape == (voxels.shape[0], 4)
        assert torch.allclose(out.double().cpu(), ref[:voxels.shape[0]].cpu(), atol=4e-3)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        out, native = launched(monkeypatch, lambda: spnn.mean_voxel_features(dual, counts))
        tangent = torch.autograd.forward_ad.unpack_dual(out).tangent
        assert not native and torch.allclose(tangent, 5.0 / counts.float()[:, None].expand(50, 4))
    out = torch.func.vmap(lambda v: spnn.mean_voxel_features(v, counts))(x[None].expand(3, -1, -1, -1))
    assert torch.allclose(out[2].double(), ref, atol=1e-5)


def test_captured(monkeypatch):
    import torch
    from mluop_hip import nn as spnn
    x = torch.randn(300, 5, 4, device="cuda")
    counts = torch.randint(1, 6, (300,), device="cuda", dtype=torch.int32)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        spnn.mean_voxel_features(x, counts)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = spnn.mean_voxel_features(x, counts)
    torch.cuda.synchronize()
    for _ in range(3):
        x.copy_(torch.randn_like(x))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, spnn.mean_voxel_features(x, counts))
