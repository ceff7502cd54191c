"""What a user of this framework has it do, as cases that can be timed and checked.

Every case goes through ``spconv_triton.pytorch`` (modules, ``ops`` and ``PointToVoxel``).  The sizes,
clouds and networks are those of ``bench.py`` and ``bench_configs.py``; ``draw`` varies them.  Kinds:

* ``layer``: the eval forward of one submanifold convolution, with its rulebook held by an
  ``indice_key`` (as the layers that share one hold it) or built in the pass (``held`` false);
* ``train``: one submanifold layer's training step (rulebook, forward, gradients of the input, the
  weight and the bias), under fp16 autocast with fp32 parameters or in the parameters' own type;
* ``updown``: a strided convolution and the inverse convolution that shares its key, training step;
* ``pool``: max pooling, forward and backward, with its tables built in the pass;
* ``rulebook``: the implicit-GEMM pair tables with sorted masks, by the public op;
* ``encoder``: a whole LiDAR voxel encoder in fp16 eval, all rulebooks built in the pass;
* ``voxelize``: a point cloud to voxels.

Clouds: ``uniform`` cells; ``surface`` (spheres and planes in a cube); ``lidar`` (a ground plane with
range fall-off and boxes); ``urban`` (road, walls, boxes); ``drift`` (a surface moving through 64 time
steps, 4-D).  Rows come in ascending order of their linear key, as a sorting voxeliser emits them.
Where the number of output rows follows from the cloud (strided tables, pooling, the encoder), a case
has one cloud, kept off the borders, which a seed mirrors and shifts by whole strides, so that every
seed has as many outputs; elsewhere each seed draws its own.
"""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "spconv-triton_amd"))

GRIDS = {"lidar": (41, 1600, 1408), "urban": (128, 2048, 2048), "drift": (64, 512, 512, 512)}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "tf32": torch.float32}

# VoxelBackBone8x-style encoder: (kind, in, out, kernel, stride, padding, key), each with BatchNorm + ReLU
ENCODER = [
    ("subm", 4, 16, 3, 1, 1, "subm1"),
    ("conv", 16, 32, 3, 2, 1, "spconv2"),
    ("subm", 32, 32, 3, 1, 1, "subm2"),
    ("subm", 32, 32, 3, 1, 1, "subm2"),
    ("conv", 32, 64, 3, 2, 1, "spconv3"),
    ("subm", 64, 64, 3, 1, 1, "subm3"),
    ("subm", 64, 64, 3, 1, 1, "subm3"),
    ("conv", 64, 64, 3, 2, (0, 1, 1), "spconv4"),
    ("subm", 64, 64, 3, 1, 1, "subm4"),
    ("subm", 64, 64, 3, 1, 1, "subm4"),
    ("conv", 64, 128, (3, 1, 1), (2, 1, 1), 0, "spconv_down2"),
]

# 70.4 m x 80 m x 4.1 m at 5 x 5 x 10 cm: the LiDAR grid's cells
VOXEL_SIZE = [0.05, 0.05, 0.1]
POINT_RANGE = [0.0, -40.0, -3.0, 70.4, 40.0, 1.1]


def listed():
    return [
        # the smallest call: a 2,000-voxel fp32 layer with a new rulebook every pass, where host
        # latency and launches count
        {"name": "subm16_f32_2k", "kind": "layer", "cloud": "uniform", "grid": 64, "n": 2000,
         "batch": 1, "cin": 16, "cout": 16, "ksize": 3, "dtype": "f32", "held": False},
        # the headline layer: 200k surface voxels in 256^3, 64 -> 64, its rulebook shared by key
        {"name": "subm64_f16_200k", "kind": "layer", "cloud": "surface", "grid": 256, "n": 200000,
         "batch": 1, "cin": 64, "cout": 64, "ksize": 3, "dtype": "f16", "held": True},
        # a wide detector layer on a LiDAR cloud (few neighbours per voxel) in IEEE fp32
        {"name": "lidar256_f32_50k", "kind": "layer", "cloud": "lidar", "grid": 0, "n": 50000,
         "batch": 1, "cin": 256, "cout": 256, "ksize": 3, "dtype": "f32", "held": True},
        # the widest listed work: 256 -> 256 on a 400k-voxel scene in 1024^3, in bf16
        {"name": "wide256_bf16_400k", "kind": "layer", "cloud": "surface", "grid": 1024,
         "n": 400000, "batch": 1, "cin": 256, "cout": 256, "ksize": 3, "dtype": "bf16",
         "held": True},
        # 4-D sequence layer: 81 offsets, int64 keys, the Native algorithm
        {"name": "subm4d128_f16_500k", "kind": "layer", "cloud": "drift", "grid": 0, "n": 500000,
         "batch": 1, "cin": 128, "cout": 128, "ksize": 3, "dtype": "f16", "held": True},
        # a full-resolution segmentation layer's training step, batch 2 x ~120k voxels, autocast
        {"name": "train64_amp_240k", "kind": "train", "cloud": "urban", "grid": 0, "n": 120000,
         "batch": 2, "cin": 64, "cout": 64, "ksize": 3, "dtype": "f16", "amp": True},
        # a wide decoder layer's training step in bf16 (the weight gradient weighs most)
        {"name": "train256_bf16_75k", "kind": "train", "cloud": "surface", "grid": 256,
         "n": 75001, "batch": 1, "cin": 256, "cout": 128, "ksize": 3, "dtype": "bf16",
         "amp": False},
        # down and up again in a U-Net: k2 s2 convolution and its inverse, training step
        {"name": "updown64_amp_240k", "kind": "updown", "cloud": "urban", "grid": 0, "n": 120000,
         "batch": 2, "cin": 64, "cout": 128, "ksize": 2, "dtype": "f16", "amp": True},
        # max pooling between two stages of it
        {"name": "pool64_f16_212k", "kind": "pool", "cloud": "urban", "grid": 0, "n": 105942,
         "batch": 2, "cin": 64, "cout": 64, "ksize": 2, "dtype": "f16"},
        # the public pair-table op for a training rulebook, with both tables and sorted masks
        {"name": "rulebook_subm_200k", "kind": "rulebook", "cloud": "surface", "grid": 256,
         "n": 200000, "batch": 1, "ksize": 3, "stride": 1, "mode": "subm"},
        # a whole LiDAR encoder pass, 4 samples of 20k voxels
        {"name": "encoder_f16_80k", "kind": "encoder", "cloud": "lidar", "grid": 0, "n": 20000,
         "batch": 4, "dtype": "f16"},
        # a 200k-point sweep to voxels, before any network
        {"name": "voxelize_200k", "kind": "voxelize", "n": 200000, "max_voxels": 150000,
         "max_points": 5, "features": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cloud(rng, lo, hi):
    """A cloud of lo..hi voxels in all (log-uniform; odd counts among them)."""
    cloud = rng.choice(["surface", "surface", "lidar", "urban", "uniform"])
    n, batch, grid = _log(rng, lo, hi), rng.choice([1, 1, 2, 4]), 0
    if cloud in ("surface", "uniform"):
        grid = 64 if n <= 20000 else 256 if n <= 250000 else 1024
        if grid == 64 and cloud == "surface":
            grid = 128
    return {"cloud": cloud, "grid": grid, "n": max(500, n // batch), "batch": batch}


def _widths(rng, rows, most):
    """(cin, cout) of the widths networks use, some no power of two, rows * cin * cout <= most."""
    widths = [16, 20, 32, 40, 48, 64, 96, 128, 160, 256]
    while True:
        cin, cout = rng.choice([3, 4] + widths), rng.choice(widths)
        if rows * cin * cout <= most:
            return cin, cout


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "train", "train", "updown", "pool", "rulebook",
                       "encoder", "voxelize"])
    if kind == "voxelize":
        n = _log(rng, 20000, 400000)
        return {"kind": kind, "n": n, "max_voxels": rng.choice([n // 8, n // 2, n]),
                "max_points": rng.choice([5, 10, 32]), "features": rng.choice([3, 4, 5])}
    if kind == "encoder":
        return {"kind": kind, "cloud": "lidar", "grid": 0, "n": _log(rng, 3000, 20000),
                "batch": rng.choice([1, 2, 3, 4]), "dtype": "f16"}
    if kind == "rulebook":
        mode = rng.choice(["subm", "subm", "strided", "transposed"])
        case = {"kind": kind, **_cloud(rng, 2000, 400000 if mode == "subm" else 100000),
                "mode": mode, "stride": 1 if mode == "subm" else 2,
                "ksize": rng.choice([3, 3, 5]) if mode == "subm" else rng.choice([2, 3])}
        if case["ksize"] == 5:
            case["n"] = min(case["n"], 50001)
        return case
    if kind == "pool":
        cin = rng.choice([16, 20, 32, 48, 64, 128])
        return {"kind": kind, **_cloud(rng, 2000, 240000), "cin": cin, "cout": cin,
                "ksize": rng.choice([2, 2, 3]), "dtype": rng.choice(["f16", "f16", "bf16", "f32"])}
    case = {"kind": kind, **_cloud(rng, 2000, 400000 if kind == "layer" else 240000)}
    # up to ten neighbours per voxel; fp32 products cost sixteen times the 16-bit ones
    most = 400000 * 64 * 64 if kind == "layer" else 240000 * 64 * 64
    dtype = rng.choice(["f16", "f16", "bf16", "f32", "tf32"])
    most //= 4 if dtype == "f32" else 2 if dtype == "tf32" else 1
    cin, cout = _widths(rng, case["n"] * case["batch"], most)
    case.update(cin=cin, cout=cout, dtype=dtype, ksize=3)
    if kind == "layer":
        case["held"] = rng.random() < 0.6
    else:
        case["amp"] = dtype == "f16" and rng.random() < 0.7
        if kind == "updown":
            case["ksize"] = rng.choice([2, 3])
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


class _Rng:
    """Seeded random numbers on the device."""

    def __init__(self, seed):
        self.dev = _device()
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed) * 7919 + 17)
        self.host = np.random.default_rng(int(seed))

    def uniform(self, lo, hi, *shape):
        u = torch.rand(*shape, generator=self.g, device=self.dev, dtype=torch.float64)
        return u * (hi - lo) + lo

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=self.dev)


def shape_of(case):
    if case["cloud"] in GRIDS:
        return list(GRIDS[case["cloud"]])
    return [case["grid"]] * 3


def _keys(points, shape, margin=0):
    """Unique linear keys of the points inside the grid, ``margin`` cells off the borders of its
    last two dimensions."""
    p = points.floor().to(torch.int64)
    low = torch.zeros(len(shape), dtype=torch.int64, device=p.device)
    low[-2:] = margin
    top = torch.tensor(shape, device=p.device) - low
    p = p[((p >= low) & (p < top)).all(1)]
    key = p[:, 0]
    for d in range(1, len(shape)):
        key = key * shape[d] + p[:, d]
    return torch.unique(key)


def _surface_points(r, grid):
    parts = []
    for _ in range(16):
        if r.host.random() < 0.5:
            c = torch.from_numpy(r.host.uniform(0.15, 0.85, 3) * grid).to(r.dev)
            d = r.normal(60000, 3).double()
            parts.append(c + r.host.uniform(0.04, 0.2) * grid * d / d.norm(dim=1, keepdim=True))
        else:
            q, _ = np.linalg.qr(r.host.standard_normal((3, 3)))
            c = torch.from_numpy(r.host.uniform(0.2, 0.8, 3) * grid).to(r.dev)
            uv = torch.from_numpy(np.ascontiguousarray(q[:2])).to(r.dev)
            half = float(r.host.uniform(0.05, 0.3) * grid)
            parts.append(c + r.uniform(-half, half, 60000, 2) @ uv)
    return torch.cat(parts)


def _boxes(r, count, points, lo, hi, floor):
    """Points on the faces of ``count`` boxes with extents lo..hi; ``floor``: they stand on it."""
    parts = []
    for _ in range(count):
        ext = r.host.uniform(lo, hi)
        face = r.uniform(-0.5, 0.5, points, 3)
        axis = torch.randint(0, 3, (points,), generator=r.g, device=r.dev)
        at = torch.arange(points, device=r.dev)
        face[at, axis] = torch.sign(face[at, axis]) * 0.5
        c = r.host.uniform(0, 1, 3) * (np.array(GRIDS["urban" if floor else "lidar"]) - 1)
        c[0] = 5 + ext[0] / 2 if floor else r.host.uniform(4, GRIDS["lidar"][0] - 8)
        parts.append(face * torch.from_numpy(ext).to(r.dev) + torch.from_numpy(c).to(r.dev))
    return parts


def _lidar_points(r):
    z, y, x = GRIDS["lidar"]
    p = r.uniform(0, 1, 200000, 3) * torch.tensor([2.0, y, x], device=r.dev, dtype=torch.float64)
    p[:, 0] += 2
    far = torch.hypot(p[:, 1] - y / 2, p[:, 2]) / math.hypot(y / 2, x)
    ground = p[r.uniform(0, 1, 200000) < 0.6 * (1 - far) ** 2]
    return torch.cat([ground] + _boxes(r, 30, 4000, np.array([4, 20, 20.0]),
                                       np.array([10, 50, 50.0]), False))


def _urban_points(r, n):
    z, y, x = GRIDS["urban"]
    road = r.uniform(0, 1, n, 3) * torch.tensor([2.0, y, x], device=r.dev, dtype=torch.float64)
    road[:, 0] += 4
    parts = [road]
    for _ in range(12):
        m = n // 8
        c, t = r.host.uniform(0, [y, x]), r.uniform(-0.5, 0.5, m) * r.host.uniform(0.1, 0.5) * x
        wall = torch.empty(m, 3, device=r.dev, dtype=torch.float64)
        wall[:, 0] = r.uniform(4, 4 + r.host.uniform(0.3, 0.9) * z, m)
        along = int(r.host.integers(1, 3))
        wall[:, along] = c[along - 1] + t
        wall[:, 3 - along] = c[2 - along]
        parts.append(wall)
    return torch.cat(parts + _boxes(r, 40, 2000, np.array([5, 20, 20.0]),
                                    np.array([15, 60, 60.0]), True))


def _sized_by_cloud(case):
    """The case's number of output rows follows from its cloud (see the top)."""
    return (case["kind"] in ("pool", "encoder")
            or case["kind"] == "rulebook" and case["mode"] != "subm")


def _moved(idx, case, seed):
    """The cloud mirrored and shifted along its last two dimensions by multiples of 8 cells, the
    encoder's stride; windows of 2 cells mirror onto each other about the middle of two."""
    host = np.random.default_rng(int(seed) + 1000003)
    idx = idx.long()
    even = case.get("ksize", 3) == 2
    for d, n in zip((2, 3), shape_of(case)[-2:]):
        if host.random() < 0.5:
            idx[:, d] = n // 8 * 8 - even - idx[:, d]
        idx[:, d] += 8 * int(host.integers(-1, 2))
    shape = shape_of(case)
    return idx[torch.argsort(_linear(idx, shape))].to(torch.int32).contiguous()


def cloud(case, seed):
    """int32 [N, ndim + 1] voxel rows (batch first), ascending by linear key."""
    if case.get("kind") and _sized_by_cloud(case):
        base = {k: case[k] for k in ("cloud", "grid", "n", "batch")}
        return _moved(cloud({**base, "margin": 16}, case["n"]), case, seed)
    shape, rows = shape_of(case), []
    for b in range(case["batch"]):
        r = _Rng(int(seed) * 64 + b)
        n = case["n"]
        if case["cloud"] == "drift":
            base = cloud({"cloud": "surface", "grid": 512, "n": max(1, n // 60), "batch": 1}, seed)
            t = torch.arange(64, device=r.dev).repeat_interleave(base.shape[0])
            c = base[:, 1:].long().repeat(64, 1) + torch.stack([t // 8, t // 16, t // 4], 1)
            keep = r.uniform(0, 1, t.shape[0]) < 0.98
            p = torch.cat([t[:, None], c.clamp(0, 511)], 1)[keep]
            keys = _keys(p.double(), shape)  # about 4 % more than n
        else:
            keys = torch.zeros(0, dtype=torch.int64, device=r.dev)
            while keys.numel() < n:
                if case["cloud"] == "uniform":
                    p = r.uniform(0, 1, 2 * n, 3) * case["grid"]
                elif case["cloud"] == "surface":
                    p = _surface_points(r, case["grid"])
                elif case["cloud"] == "lidar":
                    p = _lidar_points(r)
                else:
                    p = _urban_points(r, n)
                keys = torch.unique(torch.cat([keys, _keys(p, shape, case.get("margin", 0))]))
        pick = torch.randperm(keys.numel(), generator=r.g, device=r.dev)[:n]
        keys = torch.sort(keys[pick])[0]
        rows.append(torch.cat([torch.full_like(keys, b)[:, None], _unravel(keys, shape)], 1))
    return torch.cat(rows).to(torch.int32).contiguous()


def _unravel(keys, shape):
    cols = []
    for n in reversed(shape):
        cols.append(keys % n)
        keys = keys // n
    return torch.stack(cols[::-1], 1)


def _out_type(case):
    """The type a training layer's output has: fp16 under autocast."""
    return torch.float16 if case.get("amp") else DTYPES[case["dtype"]]


def _param_type(case):
    return torch.float32 if case.get("amp") else DTYPES[case["dtype"]]


def _tensors(case, seed, rows, out_rows=0):
    """Features and weights of a case (and the output gradient of a training step)."""
    r = _Rng(seed)
    kind, dt = case["kind"], _param_type(case)
    t = {"x": r.normal(rows, case["cin"]).to(_out_type(case))}
    if kind == "pool":
        return t, r
    nd = 4 if case["cloud"] == "drift" else 3
    kv = case["ksize"] ** nd

    def weight(cin, cout):
        bound = 1 / math.sqrt(cin * kv)
        shape = [cout] + [case["ksize"]] * nd + [cin]
        return r.uniform(-bound, bound, *shape).to(dt), r.uniform(-bound, bound, cout).to(dt)

    t["w"], t["b"] = weight(case["cin"], case["cout"])
    if kind == "updown":
        t["w2"], t["b2"] = weight(case["cout"], case["cin"])
    return t, r


def _points(case, seed):
    """A sweep: ground and box surfaces in metres, a few points out of range, features.  A case
    has one set of positions; a seed gives their order (which numbers the voxels) and features."""
    r = _Rng(case["n"])
    n, parts, have = case["n"], [], 0
    while have < n:
        parts.append(_lidar_points(r))
        have += parts[-1].shape[0]
    p = torch.cat(parts)
    p = p[torch.randperm(p.shape[0], generator=r.g, device=r.dev)[:n]]
    r = _Rng(seed)
    p = p[torch.randperm(n, generator=r.g, device=r.dev)]
    low = torch.tensor(POINT_RANGE[:3], device=r.dev, dtype=torch.float64)
    size = torch.tensor(VOXEL_SIZE, device=r.dev, dtype=torch.float64)
    pc = torch.empty(n, case["features"], device=r.dev)
    pc[:, :3] = (p.flip(1) * 1.01 * size + low).float()
    if case["features"] > 3:
        pc[:, 3:] = r.uniform(0, 1, n, case["features"] - 3).float()
    return pc


def _build(case):
    import spconv_triton.pytorch as spconv

    k, cin, cout = case["ksize"], case.get("cin"), case.get("cout")
    if case["kind"] == "pool":
        return spconv.SparseMaxPool3d(k, 2, padding=0 if k == 2 else 1, indice_key="p")
    if case["kind"] == "updown":
        return spconv.SparseSequential(
            spconv.SparseConv3d(cin, cout, k, stride=2, padding=0 if k == 2 else 1,
                                indice_key="d"),
            spconv.SparseInverseConv3d(cout, cin, k, indice_key="d"))
    cls = spconv.SubMConv4d if case["cloud"] == "drift" else spconv.SubMConv3d
    return cls(cin, cout, k, padding=k // 2, indice_key="s")


def _encoder(seed):
    """The encoder's modules and, per layer, (weight, BatchNorm scale, shift, mean, variance)."""
    import spconv_triton.pytorch as spconv

    r, mods, params = _Rng(seed + 1), [], []
    for kind, cin, cout, k, stride, pad, key in ENCODER:
        if kind == "subm":
            conv = spconv.SubMConv3d(cin, cout, k, padding=pad, bias=False, indice_key=key)
        else:
            conv = spconv.SparseConv3d(cin, cout, k, stride=stride, padding=pad, bias=False,
                                       indice_key=key)
        bn = torch.nn.BatchNorm1d(cout)
        bound = math.sqrt(6.0 / (cin * 5))
        w = r.uniform(-bound, bound, *conv.weight.shape)
        stats = [r.uniform(0.8, 1.2, cout), r.uniform(-0.2, 0.2, cout), r.uniform(-0.1, 0.1, cout),
                 r.uniform(0.5, 1.5, cout)]
        with torch.no_grad():
            conv.weight.copy_(w)
            for to, v in zip((bn.weight, bn.bias, bn.running_mean, bn.running_var), stats):
                to.copy_(v)
        mods += [conv, bn, torch.nn.ReLU()]
        params.append([v.half() for v in [w] + stats])
    return spconv.SparseSequential(*mods).to(_device()).half().eval(), params


def _strided_geometry(case):
    k = case["ksize"]
    return k, 0 if (k == 2 or case.get("mode") == "transposed") else 1


def prepare(case, seed):
    import spconv_triton.pytorch as spconv

    kind = case["kind"]
    state = {"case": dict(case)}
    if kind == "voxelize":
        from spconv_triton.pytorch.utils import PointToVoxel

        state["points"] = _points(case, seed)
        state["gen"] = PointToVoxel(VOXEL_SIZE, POINT_RANGE, case["features"], case["max_voxels"],
                                    case["max_points"], device=_device())
        return state
    idx = cloud(case, seed)
    state.update(idx=idx, shape=shape_of(case))
    if kind == "rulebook":
        return state
    if kind == "encoder":
        state["net"] = _encoder(seed)[0]
        state["x"] = _Rng(seed).uniform(0, 1, idx.shape[0], 4).half()
        return state
    t, r = _tensors(case, seed, idx.shape[0])
    state["x"] = t["x"]
    net = _build(case).to(_device())
    if kind != "pool":
        net = net.to(_param_type(case))
        with torch.no_grad():
            convs = [net] if kind != "updown" else [net[0], net[1]]
            for conv, w, b in zip(convs, ("w", "w2"), ("b", "b2")):
                conv.weight.copy_(t[w])
                conv.bias.copy_(t[b])
    state["net"] = net.eval() if kind == "layer" else net.train()
    if kind == "layer":
        if case["held"]:
            with torch.no_grad():
                y = net(spconv.SparseConvTensor(t["x"], idx, state["shape"], case["batch"]))
            state["rulebook"] = y.indice_dict
        return state
    # the gradient that the layers above send back: as many rows as the output has
    rows = idx.shape[0]
    if kind == "pool":
        rows = _strided_table(idx.long(), state["shape"], case["batch"], [case["ksize"]] * 3,
                              [2] * 3, [0 if case["ksize"] == 2 else 1] * 3)[0].shape[0]
    width = case["cin"] if kind == "updown" else case["cout"]
    state["grad"] = r.normal(rows, width).to(_out_type(case))
    return state


def run(state):
    import spconv_triton.pytorch as spconv

    case = state["case"]
    kind = case["kind"]
    if kind == "voxelize":
        return list(state["gen"].generate_voxel_with_id(state["points"]))
    if kind == "rulebook":
        from spconv_triton.core import ConvAlgo
        from spconv_triton.pytorch import ops

        k, pad = _strided_geometry(case)
        subm = case["mode"] == "subm"
        many = k ** 3 > 32
        if many:  # larger windows run the Native algorithm, as the modules choose
            return list(ops.get_indice_pairs(
                state["idx"], case["batch"], state["shape"], ConvAlgo.Native, [k] * 3,
                [case["stride"]] * 3, [k // 2 if subm else pad] * 3, [1] * 3, [0] * 3, subm,
                case["mode"] == "transposed"))
        res = ops.get_indice_pairs_implicit_gemm(
            state["idx"], case["batch"], state["shape"], ConvAlgo.MaskImplicitGemm, [k] * 3,
            [case["stride"]] * 3, [k // 2 if subm else pad] * 3, [1] * 3, [0] * 3, subm,
            case["mode"] == "transposed", is_train=True)
        return [list(v) if isinstance(v, (list, tuple)) else v for v in res[:8]]
    if kind == "encoder":
        with torch.no_grad():
            y = state["net"](spconv.SparseConvTensor(state["x"], state["idx"], state["shape"],
                                                     case["batch"]))
        return [y.features, y.indices]
    if kind == "layer":
        with _tf32(case), torch.no_grad():
            y = state["net"](spconv.SparseConvTensor(state["x"], state["idx"], state["shape"],
                                                     case["batch"],
                                                     indice_dict=state.get("rulebook")))
        return [y.features]
    x = state["x"].detach().requires_grad_(True)
    net = state["net"]
    params = [p for p in net.parameters()]
    with _tf32(case):
        with torch.autocast("cuda", dtype=torch.float16, enabled=bool(case.get("amp"))):
            y = net(spconv.SparseConvTensor(x, state["idx"], state["shape"], case["batch"]))
        grads = torch.autograd.grad(y.features, [x] + params, state["grad"])
    return [y.features.detach()] + list(grads)


class _tf32:
    """SPCONV_ALLOW_TF32 as a program that asks for TF32 sets it."""

    def __init__(self, case):
        self.on = case["dtype"] == "tf32"

    def __enter__(self):
        if self.on:
            from spconv_triton import constants

            self.before = constants.SPCONV_ALLOW_TF32
            constants.SPCONV_ALLOW_TF32 = True

    def __exit__(self, *exc):
        if self.on:
            from spconv_triton import constants

            constants.SPCONV_ALLOW_TF32 = self.before


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------

def _linear(c, shape):
    """Keys of int64 rows [b, c0, c1, ...]."""
    key = c[:, 0]
    for d, n in enumerate(shape):
        key = key * n + c[:, d + 1]
    return key


def _offsets(ksize):
    grids = torch.meshgrid(*[torch.arange(k) for k in ksize], indexing="ij")
    return torch.stack([g.reshape(-1) for g in grids], 1).tolist()


def _find(keys, wanted):
    """Rows of ``wanted`` in the ascending ``keys`` (-1: absent)."""
    at = torch.searchsorted(keys, wanted).clamp(max=keys.numel() - 1)
    return torch.where(keys[at] == wanted, at, torch.full_like(at, -1))


def _subm_pairs(idx, shape, ksize):
    """Per offset, (input rows, output rows) of a submanifold layer."""
    keys = _linear(idx, shape)
    order = torch.argsort(keys)
    keys = keys[order]
    top = torch.tensor(shape, device=idx.device)
    for off in _offsets(ksize):
        c = idx.clone()
        c[:, 1:] += torch.tensor([o - k // 2 for o, k in zip(off, ksize)], device=idx.device)
        ok = ((c[:, 1:] >= 0) & (c[:, 1:] < top)).all(1)
        row = _find(keys, _linear(c, shape))
        out = torch.nonzero(ok & (row >= 0)).view(-1)
        yield order[row[out]], out


def _strided_table(idx, shape, batch, ksize, stride, pad):
    """(output rows [b, ...] ascending, output shape, per offset (input rows, output rows))."""
    out_shape = [(n + 2 * p - k) // s + 1 for n, p, k, s in zip(shape, pad, ksize, stride)]
    st = torch.tensor(stride, device=idx.device)
    top = torch.tensor(out_shape, device=idx.device)
    cand = []
    for off in _offsets(ksize):
        c = idx[:, 1:] + torch.tensor(pad, device=idx.device) - torch.tensor(off,
                                                                             device=idx.device)
        ok = ((c >= 0) & (c % st == 0)).all(1)
        q = c // st
        ok &= (q < top).all(1)
        rows = torch.nonzero(ok).view(-1)
        cand.append((rows, _linear(torch.cat([idx[rows, :1], q[rows]], 1), out_shape)))
    keys = torch.unique(torch.cat([k for _, k in cand]))
    vol = int(np.prod(out_shape))
    out = torch.cat([(keys // vol)[:, None], _unravel(keys % vol, out_shape)], 1)
    return out, out_shape, [(rows, torch.searchsorted(keys, k)) for rows, k in cand]


def _conv(x, w, pairs, n_out):
    """y[out] += x[in] W[k]^T over the pairs of every offset; x float64, w [K, kv, C] float64."""
    y = torch.zeros(n_out, w.shape[0], dtype=torch.float64, device=x.device)
    for k, (i, o) in enumerate(pairs):
        if i.numel():
            y.index_add_(0, o, x[i] @ w[:, k].T)
    return y


def _conv_grads(x, w, g, pairs):
    dx, dw = torch.zeros_like(x), torch.zeros_like(w)
    for k, (i, o) in enumerate(pairs):
        if i.numel():
            dx.index_add_(0, i, g[o] @ w[:, k])
            dw[:, k] = g[o].T @ x[i]
    return dx, dw


def exact(case, seed):
    kind = case["kind"]
    if kind in ("voxelize", "rulebook"):
        return None  # copies of inputs and whole numbers
    idx, shape = cloud(case, seed).long(), shape_of(case)
    if kind == "encoder":
        x = _Rng(seed).uniform(0, 1, idx.shape[0], 4).half().double()
        known = {}
        for (lk, cin, cout, k, stride, pad, key), p in zip(ENCODER, _encoder(seed)[1]):
            w, scale, shift, mean, var = [v.double().to(x.device) for v in p]
            k3, s3, p3 = [[v] * 3 if isinstance(v, int) else list(v) for v in (k, stride, pad)]
            if lk == "subm":
                pairs = known.setdefault(key, list(_subm_pairs(idx, shape, k3)))
                y = _conv(x, w.reshape(cout, -1, cin), pairs, idx.shape[0])
            else:
                idx, shape, pairs = _strided_table(idx, shape, case["batch"], k3, s3, p3)
                y = _conv(x, w.reshape(cout, -1, cin), pairs, idx.shape[0])
            x = torch.relu((y - mean) / torch.sqrt(var + 1e-5) * scale + shift)
        return [x, None]
    t, r = _tensors(case, seed, idx.shape[0])
    x, k = t["x"].double(), case["ksize"]
    nd, pad = len(shape), 0 if k == 2 else 1
    if kind == "layer":
        w = t["w"].double().reshape(case["cout"], -1, case["cin"])
        return [_conv(x, w, _subm_pairs(idx, shape, [k] * nd), idx.shape[0]) + t["b"].double()]
    if kind == "train":
        w = t["w"].double().reshape(case["cout"], -1, case["cin"])
        pairs = list(_subm_pairs(idx, shape, [k] * nd))
        g = r.normal(idx.shape[0], case["cout"]).to(_out_type(case)).double()
        dx, dw = _conv_grads(x, w, g, pairs)
        return [_conv(x, w, pairs, idx.shape[0]) + t["b"].double(), dx,
                dw.reshape(t["w"].shape), g.sum(0)]
    out, _, pairs = _strided_table(idx, shape, case["batch"], [k] * 3, [2] * 3, [pad] * 3)
    if kind == "pool":
        g = r.normal(out.shape[0], case["cin"]).to(_out_type(case)).double()
        y = torch.zeros(out.shape[0], case["cin"], dtype=torch.float64, device=x.device)
        for i, o in pairs:
            y.index_reduce_(0, o, x[i], "amax")
        dx = torch.zeros_like(x)
        for i, o in pairs:
            dx.index_add_(0, i, torch.where(x[i] == y[o], g[o], torch.zeros_like(g[o])))
        return [y, dx]
    g = r.normal(idx.shape[0], case["cin"]).to(_out_type(case)).double()
    w = t["w"].double().reshape(case["cout"], -1, case["cin"])
    w2 = t["w2"].double().reshape(case["cin"], -1, case["cout"])
    back = [(o, i) for i, o in pairs]
    mid = _conv(x, w, pairs, out.shape[0]) + t["b"].double()
    y = _conv(mid, w2, back, idx.shape[0]) + t["b2"].double()
    dmid, dw2 = _conv_grads(mid, w2, g, back)
    dx, dw = _conv_grads(x, w, dmid, pairs)
    return [y, dx, dw.reshape(t["w"].shape), dmid.sum(0), dw2.reshape(t["w2"].shape), g.sum(0)]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _size(case):
    return 2 if case["dtype"] in ("f16", "bf16") else 4


def work(case):
    """Inputs read once and outputs written once; two operations per product of a pair."""
    kind = case["kind"]
    if kind == "voxelize":
        n, f = case["n"], case["features"]
        out = min(n, case["max_voxels"])
        return {"bytes": 4 * n * f + out * (4 * case["max_points"] * f + 16) + 8 * n, "flops": 0}
    idx, shape = cloud(case, 1).long(), shape_of(case)
    n, nd = idx.shape[0], len(shape)
    if kind == "encoder":
        nbytes, flops, known = 2 * n * 4 + 4 * n * 4, 0, {}
        for lk, cin, cout, k, stride, pad, key in ENCODER:
            k3, s3, p3 = [[v] * 3 if isinstance(v, int) else list(v) for v in (k, stride, pad)]
            if lk == "subm":
                if key not in known:
                    known[key] = sum(i.numel() for i, _ in _subm_pairs(idx, shape, k3))
                pairs = known[key]
            else:
                idx, shape, lists = _strided_table(idx, shape, case["batch"], k3, s3, p3)
                pairs = sum(i.numel() for i, _ in lists)
            nbytes += 2 * int(np.prod(k3)) * cin * cout
            flops += 2 * pairs * cin * cout
        return {"bytes": nbytes + idx.shape[0] * (2 * 128 + 16), "flops": flops}
    k = case["ksize"]
    kv = k ** nd
    if kind == "rulebook":
        table = 4 * n * (nd + 1)
        if case["mode"] == "subm":
            return {"bytes": table + 4 * n * (2 * kv if kv > 32 else 2 * kv + 2), "flops": 0}
        if case["mode"] == "strided":
            m = _strided_table(idx, shape, case["batch"], [k] * 3, [2] * 3,
                               [_strided_geometry(case)[1]] * 3)[0].shape[0]
        else:
            m = torch.unique(torch.cat([_linear(torch.cat([idx[:, :1], idx[:, 1:] * 2 + torch.tensor(
                off, device=idx.device)], 1), [2 * s + k for s in shape])
                for off in _offsets([k] * 3)])).numel()
        return {"bytes": table + 4 * m * 4 + 4 * kv * (n + m) + 8 * (n + m), "flops": 0}
    cin, cout, e = case["cin"], case["cout"], _size(case)
    if kind in ("layer", "train"):
        pairs = sum(i.numel() for i, _ in _subm_pairs(idx, shape, [k] * nd))
        rows_in, rows_out, w = n * cin, n * cout, kv * cin * cout
        if kind == "layer":
            return {"bytes": e * (rows_in + rows_out + w) + 4 * n * (nd + 1),
                    "flops": 2 * pairs * cin * cout}
        return {"bytes": e * (2 * rows_in + 2 * rows_out + 2 * w) + 4 * n * (nd + 1),
                "flops": 6 * pairs * cin * cout}
    out, _, lists = _strided_table(idx, shape, case["batch"], [k] * 3, [2] * 3,
                                   [0 if k == 2 else 1] * 3)
    pairs, m = sum(i.numel() for i, _ in lists), out.shape[0]
    if kind == "pool":
        return {"bytes": e * cin * (2 * n + 2 * m) + 16 * (n + m), "flops": 0}
    return {"bytes": e * (4 * n * cin + 4 * kv * cin * cout) + 16 * n,
            "flops": 12 * pairs * cin * cout}


def tolerance(case):
    """Whole numbers and copies are the same; sums differ by the rounding of their type."""
    kind = case["kind"]
    if kind in ("voxelize", "rulebook"):
        return "exact"
    if kind == "encoder":  # eleven layers rounded to fp16 after each of three steps
        return {"rel": 4e-3}
    if kind == "pool":  # copies, and sums of a few gradients
        return "exact" if case["ksize"] == 2 else {"rel": {"f16": 1e-3, "bf16": 8e-3}.get(
            case["dtype"], 1e-6)}
    if case["dtype"] == "f16":
        return {"rel": 2e-3}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1e-4 if case["dtype"] == "tf32" else 1e-5}
