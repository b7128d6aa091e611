"""Performance cases of the sparse-convolution stack: what a detection or segmentation program has it do.

    points --Voxelization--> voxels --SparseTensor--> sparse layers --> features (and gradients)

Every case calls the public Python entry points (`mluop_hip.nn` for layers, `mluop_hip` for the
point scatter), so the time of a pass holds everything a caller pays for: the rulebook of a new
set of coordinates, the copy of its pair counts to the host, workspaces, launches, autograd.

Kinds of cases
  voxelize   hard voxelization of one point cloud (the first step of every inference and training step)
  scatter    dynamic voxelization: features of points reduced per voxel, mean (inference) or max with
             its gradient (training)
  subm       one submanifold layer
  strided    one strided layer, 3x3x3 or 2x2x2, stride 2
  updown     a strided 2x2x2 layer and the inverse layer that leads back to its input cells (one level
             of a segmentation U-Net)
  encoder    a whole sparse encoder on voxels: a submanifold stage, three times (strided layer, two
             submanifold layers), ReLU behind each layer
  pipeline   from points to encoder features: voxelization, mean of the points, ordering, encoder;
             what an inference program runs for each frame

Layers run as inference (`train` false: forward only) or as a training step (`train` true: forward,
gradient of the input features and of the filter)."""
import math
import os
import sys
import zlib

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "mlu-ops_amd", "python")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import mluop_hip as ops  # noqa: E402
from mluop_hip import datagen  # noqa: E402
from mluop_hip import nn as spnn  # noqa: E402

# Spatial extents (D, H, W) that layers see
SPACES = {
    "small": (40, 400, 352),      # a coarse grid or a crop
    "lidar": (41, 1600, 1408),    # first stage of a detection encoder, 5 cm cells
    "wide": (41, 1440, 1440),     # the same for a cloud around the vehicle
    "stage": (11, 360, 360),      # third stage of such an encoder
    "indoor": (64, 1024, 1024),   # scanned surfaces
}

# Pairs a row has with a 3x3x3 submanifold kernel on each kind of cloud (measured on the generators;
# used for `work` only).  "scene" and "surface" depend on how far the cloud fills its grid.
PAIRS_PER_ROW = {"uniform": 1.1, "clustered": 2.2, "surface": 2.0, "scene": 11.0}

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def listed():
    return [
        # One sweep of a small sensor, the voxel grid of a detection model: the smallest voxelizer call.
        dict(name="voxelize_sweep", kind="voxelize", points=23_417, features=4, spread="scan",
             max_points=5, max_voxels=16_000),
        # Several sweeps in one cloud, as the upstream benchmark of this repository has them.
        dict(name="voxelize_sweeps", kind="voxelize", points=1_200_000, features=4, spread="uniform",
             max_points=5, max_voxels=150_000),
        # Dynamic voxelization behind a point network in training: wide features, maximum, gradient.
        dict(name="scatter_max_train", kind="scatter", points=400_000, features=32, spread="scan", reduce="max", train=True),
        # First layer of a network on a small crop, rows in the order of a voxelizer: launches and latency.
        dict(name="subm_first_small", kind="subm", cloud="uniform", space="small", batch=1, rows=3_001, order="mixed",
             kernel=3, ci=5, co=16, dtype="float32", train=True),
        # Mid-size submanifold layer of a detection network, two clouds in a batch, bf16 inference, odd width.
        dict(name="subm_48_infer", kind="subm", cloud="clustered", space="lidar", batch=2, rows=59_998, order="cell",
             kernel=3, ci=48, co=48, dtype="bfloat16", train=False),
        # The submanifold layer of this repository's headline benchmark, as a training step.
        dict(name="subm_64_train", kind="subm", cloud="clustered", space="lidar", batch=1, rows=120_000, order="cell",
             kernel=3, ci=64, co=64, dtype="float16", train=True),
        # Submanifold layer on the filled surfaces of a driving scene, deep stage width, as a training step.
        dict(name="subm_128_scene_train", kind="subm", cloud="scene", space="wide", batch=4, rows=248_636, order="cell",
             kernel=3, ci=128, co=128, dtype="float16", train=True),
        # Large kernel on scanned surfaces, inference.
        dict(name="subm_5x5x5_infer", kind="subm", cloud="surface", space="indoor", batch=1, rows=400_000, order="cell",
             kernel=5, ci=128, co=128, dtype="float16", train=False),
        # Strided layer of a detection network on four clouds in voxelizer order, as a training step.
        dict(name="strided_64_train", kind="strided", cloud="clustered", space="lidar", batch=4, rows=120_000, order="mixed",
             kernel=3, ci=64, co=64, dtype="bfloat16", train=True),
        # One level of a segmentation U-Net in fp32, down and up again, as a training step.
        dict(name="updown_fp32_train", kind="updown", cloud="surface", space="indoor", batch=1, rows=200_000, order="cell",
             kernel=2, ci=64, co=96, dtype="float32", train=True),
        # A frame of a detection program from points to encoder features.
        dict(name="pipeline_infer", kind="pipeline", points=180_000, features=5, spread="scan", max_points=10,
             max_voxels=120_000, base=16, dtype="float16"),
        # A training step of the same encoder on voxels (the `backbone` workload of bench.py).
        dict(name="encoder_train", kind="encoder", cloud="clustered", space="lidar", rows=120_000, features=5, base=16,
             dtype="float16", train=True),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["voxelize", "voxelize", "scatter", "scatter", "subm", "subm", "subm", "strided", "updown",
                       "encoder", "pipeline"])
    if kind == "voxelize":
        return dict(kind=kind, points=_log(rng, 5_000, 1_200_000), features=rng.choice([3, 4, 5, 6]),
                    spread=rng.choice(["scan", "uniform"]), max_points=rng.choice([1, 5, 10, 20, 35]),
                    max_voxels=rng.choice([12_000, 16_000, 40_000, 60_000, 120_000, 150_000]))
    if kind == "scatter":
        reduce = rng.choice(["mean", "max"])
        features = rng.choice([3, 4, 5, 9, 16, 32, 64])
        most = min(1_000_000, 20_000_000 // features)
        return dict(kind=kind, points=_log(rng, 5_000, most), features=features, spread=rng.choice(["scan", "uniform"]),
                    reduce=reduce, train=reduce == "max" and rng.random() < 0.5)
    if kind == "encoder":
        return dict(kind=kind, cloud=rng.choice(["clustered", "scene"]), space=rng.choice(["lidar", "wide"]),
                    rows=_log(rng, 8_000, 120_000), features=rng.choice([3, 4, 5]), base=16,
                    dtype=rng.choice(["float16", "bfloat16"]), train=rng.random() < 0.5)
    if kind == "pipeline":
        return dict(kind=kind, points=_log(rng, 15_000, 400_000), features=rng.choice([4, 5]), spread="scan",
                    max_points=rng.choice([5, 10]), max_voxels=rng.choice([16_000, 40_000, 120_000]), base=16,
                    dtype=rng.choice(["float16", "bfloat16"]))
    dtype = rng.choice(["float16", "float16", "bfloat16", "float32"])
    space = rng.choice(sorted(SPACES))
    cloud = rng.choice(["uniform", "clustered", "surface", "scene"])
    batch = rng.choice([1, 1, 2, 4])
    # (half of a coarse grid at most: fuller grids belong to dense convolutions)
    top = {"small": 100_000, "stage": 150_000}.get(space, 250_000)
    if dtype == "float32":
        top = min(top, 150_000)
    rows = _log(rng, 1_500, top)
    if kind == "subm":
        ci = rng.choice([4, 5, 16, 24, 32, 48, 64, 96, 128])
        co = rng.choice([16, 32]) if ci < 16 else ci
        kernel = rng.choice([3, 3, 3, 5])
    else:
        ci = rng.choice([16, 24, 32, 48, 64, 96])
        co = rng.choice([ci, min(2 * ci, 128)])
        kernel = 2 if kind == "updown" else rng.choice([3, 3, 2])
    return dict(kind=kind, cloud=cloud, space=space, batch=batch, rows=rows, order=rng.choice(["cell", "cell", "mixed"]),
                kernel=kernel, ci=ci, co=co, dtype=dtype, train=kernel < 5 and rng.random() < 0.6)


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


# How many cells a layer reaches depends on the coordinates.  Clouds of one case have one shape, so that
# their results have one size: the shape follows from the case, its place in the grid (a multiple of
# the encoder's total stride, inside a margin that no layer's reach leaves), the order of its rows and
# all values from the seed.
MARGIN = 64
STEP = 8


def _shape_seed(case):
    return zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode())


def _place(seed):
    rng = np.random.default_rng(seed)
    return [int(v) * STEP for v in rng.integers(1, MARGIN // STEP, 2)]


def _cloud_cells(case, seed):
    """int32 [rows, 4] distinct cells (n, d, h, w) on the GPU: ascending by cell, or in mixed order (a
    voxelizer numbers its voxels by their first point)."""
    rows, batch = case["rows"], case.get("batch", 1)
    d, h, w = SPACES[case["space"]]
    grid, shape = (batch, d, h - MARGIN, w - MARGIN), _shape_seed(case)
    if case["cloud"] == "clustered":
        idx = datagen.clustered_voxels(grid, -(-rows // batch), shape)[:rows]
    else:
        idx = getattr(datagen, case["cloud"] + "_voxels")(grid, rows, shape)
    idx[:, 2:] += np.array(_place(seed), dtype=np.int32)
    if case.get("order") == "mixed":
        idx = idx[np.random.default_rng(seed).permutation(rows)]
    return torch.from_numpy(np.ascontiguousarray(idx, dtype=np.int32)).cuda()


POINT_RANGE = (0.0, -40.0, -3.0, 70.4, 40.0, 1.0)
VOXEL_SIZE = (0.05, 0.05, 0.1)
CELLS = (1408, 1600, 40)


def _point_cells(case, seed):
    """int64 [n, 3] cells (x, y, z) of points, -1 where a point lies outside the range.  "scan": what a
    spinning sensor sees, in the order of its sweep: ground rings that thin out with the distance,
    upright faces of objects, about a tenth of the returns outside.  "uniform": strewn over the range,
    a twentieth outside."""
    n, g = case["points"], _generator(_shape_seed(case))

    def rand(m=n):
        return torch.rand(m, generator=g, device="cuda")

    wide = torch.tensor([CELLS[0] - MARGIN, CELLS[1] - MARGIN, CELLS[2]], device="cuda")
    if case["spread"] == "uniform":
        cells = (torch.rand((n, 3), generator=g, device="cuda") * wide).long()
        outside = rand() < 0.05
    else:
        azimuth = torch.sort((rand() - 0.5) * 2.2).values   # radians, as swept
        distance = 2.5 + 16.0 * torch.empty(n, device="cuda").exponential_(generator=g)
        height = -1.7 + 0.03 * torch.randn(n, generator=g, device="cuda")
        # the sweep is cut into sectors, each with an object's face at its own distance
        sector = ((azimuth + 1.1) * (300 / 2.2)).long().clamp_(0, 299)
        face = 4.0 + 45.0 * rand(300)
        on_object = rand() < 0.4
        distance = torch.where(on_object, face[sector] + 0.05 * torch.randn(n, generator=g, device="cuda"), distance)
        height = torch.where(on_object, -1.7 + 2.0 * rand(), height)
        xyz = torch.stack([distance * torch.cos(azimuth), distance * torch.sin(azimuth) + 38.4, height + 3.0], dim=1)
        cells = torch.floor(xyz / torch.tensor(VOXEL_SIZE, device="cuda")).long()
        outside = ((cells < 0) | (cells >= wide)).any(dim=1)
    y, x = _place(seed)
    cells += torch.tensor([x, y, 0], device="cuda")
    cells[outside] = -1
    return cells


def _points(case, seed):
    """float32 [n, features] points, x y z first, somewhere inside their cells; far away where they have none."""
    g = _generator(seed)
    cells = _point_cells(case, seed)
    pts = torch.rand((case["points"], case["features"]), generator=g, device="cuda")
    inside = cells.double() + 0.1 + 0.8 * pts[:, :3].double()
    pts[:, :3] = (torch.tensor(POINT_RANGE[:3], device="cuda").double() +
                  inside * torch.tensor(VOXEL_SIZE, device="cuda").double()).float()
    pts[cells[:, 0] < 0, :3] += 200.0
    return pts.contiguous()


def _encoder(features, base, dtype, seed):
    torch.manual_seed(seed)
    layers = [spnn.SubMConv3d(features, base, 3, indice_key="s1"), spnn.SubMConv3d(base, base, 3, indice_key="s1")]
    c = base
    for stage in (2, 3, 4):
        layers.append(spnn.SparseConv3d(c, 2 * c, 3, stride=2, padding=1))
        layers += [spnn.SubMConv3d(2 * c, 2 * c, 3, indice_key="s%d" % stage) for _ in range(2)]
        c *= 2
    net = spnn.SparseSequential(*[m for layer in layers for m in (layer, torch.nn.ReLU())])
    for layer in layers:   # gain of a network that has been trained: activations keep their size through the ReLUs
        layer.weight.data *= 3.0
    return net.cuda().to(dtype)


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    if kind in ("voxelize", "pipeline"):
        points = _points(case, seed)
        voxelizer = spnn.Voxelization(VOXEL_SIZE, POINT_RANGE, case["max_points"], case["max_voxels"]).cuda()
        state = dict(kind=kind, points=points, voxelizer=voxelizer)
        if kind == "pipeline":
            d, h, w = voxelizer.grid_shape()
            state.update(space=(d + 1, h, w), dtype=DTYPES[case["dtype"]],
                         net=_encoder(case["features"], case["base"], DTYPES[case["dtype"]], seed))
        return state
    if kind == "scatter":
        # voxel coordinates (z, y, x) of the points, -1 outside the range, as a dynamic voxelizer gives them
        coors = _point_cells(case, seed).flip(1).to(torch.int32).contiguous()
        feats = torch.randn((case["points"], case["features"]), generator=g, device="cuda")
        state = dict(kind=kind, handle=ops.make_handle_on_current_stream(), feats=feats, coors=coors,
                     reduce=case["reduce"], train=case["train"])
        if case["train"]:
            state["grad"] = torch.randn((case["points"], case["features"]), generator=g, device="cuda")
        return state

    dtype = DTYPES[case["dtype"]]
    batch = case.get("batch", 1)
    indices = _cloud_cells(case, seed)
    ci = case["features"] if kind == "encoder" else case["ci"]
    feats = torch.randn((case["rows"], ci), generator=g, device="cuda").to(dtype)
    torch.manual_seed(seed)
    if kind == "encoder":
        layers = [_encoder(ci, case["base"], dtype, seed)]
    elif kind == "subm":
        layers = [spnn.SubMConv3d(ci, case["co"], case["kernel"])]
    elif kind == "strided":
        layers = [spnn.SparseConv3d(ci, case["co"], case["kernel"], stride=2, padding=case["kernel"] // 2 if case["kernel"] == 3 else 0)]
    else:
        layers = [spnn.SparseConv3d(ci, case["co"], 2, stride=2, indice_key="down"),
                  spnn.SparseInverseConv3d(case["co"], ci, 2, "down")]
    layers = [layer.cuda().to(dtype) for layer in layers]
    state = dict(kind=kind, feats=feats, indices=indices, space=SPACES[case["space"]], batch=batch, layers=layers,
                 train=case["train"])
    if case["train"]:
        feats.requires_grad_(True)
        state["leaves"] = [feats] + [p for layer in layers for p in layer.parameters()]
        # the gradient that arrives from the layers behind
        with torch.no_grad():
            shape = _forward(state).features.shape
        state["grad"] = (torch.randn(shape, generator=g, device="cuda") * 0.01).to(dtype)
    return state


# ---------------------------------------------------------------------------------------------
# A pass
# ---------------------------------------------------------------------------------------------

def _forward(s):
    x = spnn.SparseTensor(s["feats"], s["indices"], s["space"], s["batch"], distinct=True)
    for layer in s["layers"]:
        x = layer(x)
    return x


def run(s):
    kind = s["kind"]
    if kind == "voxelize":
        return s["voxelizer"](s["points"])
    if kind == "pipeline":
        with torch.no_grad():
            voxels, coors, counts = s["voxelizer"](s["points"])
            feats = spnn.mean_voxel_features(voxels, counts).to(s["dtype"])
            x = s["net"](spnn.sparse_tensor_from_voxels(feats, coors, s["space"]))
        return x.features, x.indices
    if kind == "scatter":
        out = ops.dynamic_point_to_voxel_forward(s["handle"], s["feats"], s["coors"], s["reduce"])
        if not s["train"]:
            return out
        voxel_feats, voxel_coors, p2v, count, num = out
        grad = ops.dynamic_point_to_voxel_backward(s["handle"], s["grad"], s["feats"], voxel_feats, p2v, count, num)
        return out + (grad,)
    if not s["train"]:
        with torch.no_grad():
            x = _forward(s)
        return x.features, x.indices
    x = _forward(s)
    return (x.features.detach(), x.indices) + torch.autograd.grad(x.features, s["leaves"], s["grad"])


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, and how exact its results are
# ---------------------------------------------------------------------------------------------

def _layer_work(rows_in, rows_out, pairs, k, ci, co, size, train):
    """Features and filter in, result out; training: the arriving gradient in, both gradients out."""
    once = (rows_in * ci + k * ci * co + rows_out * co) * size
    return once * (2 if train else 1), 2.0 * pairs * ci * co * (3 if train else 1)


def _pairs_per_row(case):
    """Pairs per row of a submanifold layer, 3x3x3; clouds that fill more of their grid have more."""
    return PAIRS_PER_ROW[case["cloud"]]


def work(case):
    kind = case["kind"]
    if kind == "voxelize":
        # the points in; every kept point, the coordinates and the counts out (a fifth of the points share
        # their voxel with another one)
        n, v = case["points"], min(case["points"], case["max_voxels"])
        return dict(bytes=n * case["features"] * 4 + v * (case["max_points"] * case["features"] * 4 + 16), flops=0)
    if kind == "scatter":
        n, c = case["points"], case["features"]
        moved = n * (4 * c + 12) + n * (4 * c + 12 + 4 + 4)   # in: features, coordinates; out: the tables
        if case["train"]:
            moved += n * 4 * c * 2                            # the arriving gradient in, the gradient out
        return dict(bytes=moved, flops=n * c)
    size = 4 if case.get("dtype") == "float32" else 2
    if kind in ("encoder", "pipeline"):
        train = case.get("train", False)
        rows = case["rows"] if kind == "encoder" else min(case["points"] // 2, case["max_voxels"])
        # rows of the four stages and pairs per row there: a strided layer spreads sparse clouds out first
        heights, dense = (1.0, 2.2, 2.0, 1.2), (2.5, 10.0, 12.0, 16.0)
        moved, flops = rows * 16.0, 0.0
        c_in, c = case["features"], case["base"]
        for stage in range(4):
            r = rows * heights[stage]
            first = rows * heights[max(stage - 1, 0)]
            shapes = [(first, r, c_in, c)] + [(r, r, c, c)] * (1 if stage == 0 else 2)
            for rows_in, rows_out, a, b in shapes:
                pairs = r * dense[stage] if rows_in == rows_out else first * 3.4
                flops += 2.0 * pairs * a * b * (3 if train else 1)
                moved += 27 * a * b * size * (2 if train else 1)
            c_in, c = c, 2 * c
        moved += rows * case["features"] * size * (2 if train else 1) + rows * heights[3] * 8 * case["base"] * size * (2 if train else 1)
        if kind == "pipeline":
            moved += case["points"] * case["features"] * 4
        return dict(bytes=moved, flops=flops)
    rows, ci, co, train = case["rows"], case["ci"], case["co"], case["train"]
    k = case["kernel"] ** 3
    moved = rows * 16.0                                       # the coordinates
    if kind == "subm":
        pairs = rows * _pairs_per_row(case) * (1 if case["kernel"] == 3 else 2)
        m, f = _layer_work(rows, rows, pairs, k, ci, co, size, train)
    elif kind == "strided":
        out, pairs = (rows * 2.2, rows * 3.4) if case["kernel"] == 3 else (rows * 0.7, float(rows))
        m, f = _layer_work(rows, out, pairs, k, ci, co, size, train)
        moved += out * 16
    else:
        # features in, features out (the tensor between the two layers need not leave the chip's reach)
        m, f = _layer_work(rows, rows, 2.0 * rows, 2 * k, ci, co, size, train)
        m = (2 * rows * ci + 2 * k * ci * co) * size * (2 if train else 1)
    return dict(bytes=moved + m, flops=f)


def tolerance(case):
    kind = case["kind"]
    if kind == "voxelize" or (kind == "scatter" and case["reduce"] == "max"):
        return "exact"                      # whole numbers, and points copied bit for bit
    if kind == "scatter":
        return {"rel": 1e-6}                # sums of a few fp32 values
    if kind in ("encoder", "pipeline"):     # eleven layers, each rounded once: 2^-11 and 2^-8 a layer
        return {"rel": 5e-3, "max": 0.1} if case["dtype"] == "float16" else {"rel": 2e-2, "max": 0.4}
    # one rounding of fp32 sums (two layers in a row: one more)
    return {"float32": {"rel": 1e-5}, "float16": {"rel": 1e-3}, "bfloat16": {"rel": 6e-3}}[case["dtype"]]
