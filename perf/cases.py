"""What this framework is measured on: the calls that segmentation and detection programs make, from
one small object to batches of whole scans.

A case names its ``kind``:

  segment  inference of the residual U-Net (42 convolutions, norms folded) and its classifier over a
           tensor of new coordinates: every kernel map is built in the pass
  train    one training step of the same network: maps, forward, loss, backward, SGD
  detect   inference of the detection backbone over merged sweeps, maps built in the pass
  layer    one convolution over kernel maps that the program keeps, forward or forward and backward,
           in any of the three dataflows
  maps     the kernel maps of one tensor: submanifold, and the strided one below it
  points   the point-voxel stage of a point-voxel network: hashes, queries, counts, means into voxels
           and trilinear values back at the points, forward and backward
  loader   what a data loader's worker does with a batch of clouds on the host: quantise and collate

Clouds are ray-cast: a spinning sensor of ``beams`` beams above a ground plane with boxes, some range
noise, as many sweeps merged as it takes, and of those the sector that holds exactly ``voxels`` voxels,
``scans`` such clouds in a batch.  The sizes of a case therefore hold for every seed."""
import math
from functools import lru_cache

import numpy as np
import torch

import torchsparse_amd as ts
from torchsparse_amd import nn as spnn
from torchsparse_amd.backbones import SparseResUNet42, VoxelResBackBone8x
from torchsparse_amd.nn import functional as F
from torchsparse_amd.nn.utils import fuse_inference, get_kernel_offsets
from torchsparse_amd.utils.collate import sparse_collate
from torchsparse_amd.utils.quantize import sparse_quantize

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
DATAFLOWS = {"implicit": F.Dataflow.ImplicitGEMM, "gather_scatter": F.Dataflow.GatherScatter,
             "fetch_on_demand": F.Dataflow.FetchOnDemand}
CLASSES = 19
GRID = (41, 1440, 1440)  # (z, y, x) cells of the detection range, 0.2 m and 0.075 m

# ------------------------------------------------------------------------------ the cases


def listed():
    return [
        # one object or a small indoor crop in the precision networks are debugged in: launches and host work count
        dict(name="segment_object_fp32", kind="segment", scans=1, voxels=3403, beams=32, dtype="fp32"),
        # the scan of a 64-beam sensor, one at a time as a vehicle delivers them
        dict(name="segment_scan_fp16", kind="segment", scans=1, voxels=80003, beams=64, dtype="fp16"),
        # an evaluation run: four such scans in a batch
        dict(name="segment_batch_bf16", kind="segment", scans=4, voxels=80000, beams=64, dtype="bf16"),
        # training on a batch of crops
        dict(name="train_crops_bf16", kind="train", scans=4, voxels=11117, beams=64, dtype="bf16"),
        # training on whole scans
        dict(name="train_scan_fp16", kind="train", scans=1, voxels=80003, beams=64, dtype="fp16"),
        # a detector's backbone: two frames of merged sweeps of a 32-beam sensor
        dict(name="detect_frames_fp16", kind="detect", scans=2, voxels=110001, beams=32, dtype="fp16"),
        # the wide layer of a network over a large batch, forward and backward
        dict(name="layer_large_fp16", kind="layer", scans=10, voxels=82001, beams=64, voxel=0.05, cin=128, cout=128,
             kernel=3, stride=1, dtype="fp16", backward=True, dataflow="implicit"),
        # channel counts that are no multiple of anything: decorated points in, class scores out
        dict(name="layer_odd_fp32", kind="layer", scans=1, voxels=30011, beams=64, voxel=0.1, cin=23, cout=45,
             kernel=3, stride=1, dtype="fp32", backward=True, dataflow="implicit"),
        # a layer in the dataflow that older models are configured with
        dict(name="layer_pairs_fp16", kind="layer", scans=1, voxels=53077, beams=64, voxel=0.05, cin=64, cout=96,
             kernel=3, stride=1, dtype="fp16", backward=False, dataflow="gather_scatter"),
        # rows as a voxeliser that does not sort leaves them
        dict(name="maps_unsorted", kind="maps", scans=2, voxels=80003, beams=64, voxel=0.05, kernel=3, down=2,
             shuffled=True),
        # the points of a scan against its voxels, in a point-voxel network
        dict(name="points_scan_fp16", kind="points", scans=1, voxels=52001, per_voxel=2.0, beams=64, voxel=0.1,
             channels=64, dtype="fp16"),
        # a loader's worker with a batch of two scans
        dict(name="loader_scans", kind="loader", scans=2, voxels=80003, per_voxel=1.25, beams=64, voxel=0.05),
    ]


SCAN = 82_001  # voxels of the largest single cloud
MOST = {"segment": 320_000, "train": 80_003, "detect": 220_000, "layer": 820_010, "maps": 820_010, "points": 328_000,
        "loader": 160_006}  # voxels of a batch
LEAST = {"segment": 3000, "train": 3000, "detect": 4000, "layer": 500, "maps": 500, "points": 1000, "loader": 1000}


def _spread(rng, low, high):
    """A whole number from low to high, its logarithm spread evenly."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("segment", "segment", "train", "train", "detect", "layer", "layer", "layer", "maps", "maps",
                       "points", "points", "loader"))
    dtype = rng.choice(("fp16", "fp16", "bf16", "fp32"))
    # (precision costs time: no more of it than the listed networks take)
    rows = _spread(rng, LEAST[kind], MOST[kind] // (4 if dtype == "fp32" and kind in ("segment", "train") else 1))
    case = dict(kind=kind, scans=max(min(rng.randint(1, 4), rows // 1500), -(-rows // SCAN), 1))
    case["voxels"] = rows // case["scans"]
    case["beams"] = 32 if kind == "detect" else rng.choice((32, 64))
    if kind in ("layer", "maps", "points", "loader"):
        case["voxel"] = round(math.exp(rng.uniform(math.log(0.05), math.log(0.2))), 3)
    if kind in ("points", "loader"):
        case["per_voxel"] = round(rng.uniform(1.2, 4.0), 2)
        case["voxels"] = min(case["voxels"], int(SCAN * 2 / case["per_voxel"]))
    if kind in ("segment", "train", "detect", "layer", "points"):
        case["dtype"] = dtype
    if kind == "layer":
        case["dataflow"] = rng.choice(("implicit", "implicit", "gather_scatter", "fetch_on_demand"))
        case["backward"] = rng.random() < 0.5
        case["kernel"], case["stride"] = rng.choice(((3, 1), (3, 1), (3, 2), (2, 2), (5, 1)))
        # two thirds of the channel counts are ones networks are built of, the others anything
        for side in ("cin", "cout"):
            case[side] = rng.choice((16, 32, 64, 96, 128, 256)) if rng.random() < 2 / 3 else _spread(rng, 3, 200)
        # no more multiplications than the largest listed layer has
        most = (1.5e11 if case["dtype"] == "fp32" else 3.6e11) * (1 if case["backward"] else 3)
        most = min(most / (case["kernel"] ** 3 * case["cin"] * case["cout"]), rows)
        case["scans"] = max(min(case["scans"], int(most // 500)), 1)
        case["voxels"] = min(case["voxels"], int(most) // case["scans"])
    if kind == "maps":
        case["shuffled"] = rng.random() < 0.5
        case["kernel"] = rng.choice((3, 3, 5)) if rows < MOST["maps"] // 5 else 3
        case["down"] = rng.choice((2, 2, 3))
    if kind == "points":
        case["channels"] = rng.choice((4, 32, 64, 96, 128)) if rng.random() < 2 / 3 else _spread(rng, 3, 160)
    return case


# ------------------------------------------------------------------------------ clouds


def _scene(gen, device):
    """Low and high corners of thirty boxes on the ground, 5 to 55 m away."""
    def rand(low, high):
        return low + (high - low) * torch.rand(30, generator=gen, device=device)

    radius, angle = rand(5.0, 55.0), rand(0.0, 2 * math.pi)
    x, y, zero = radius * angle.cos(), radius * angle.sin(), torch.zeros(30, device=device)
    length, width, height = rand(1.5, 5.0), rand(1.5, 5.0), rand(1.0, 3.0)
    return (torch.stack((x - length / 2, y - width / 2, zero), 1),
            torch.stack((x + length / 2, y + width / 2, height), 1))


def _sweep(case, scene, at, gen, device):
    """float32 [P, 3] returns of one turn of the sensor, 1.8 m above the ground at x = ``at`` metres."""
    low, high = scene
    azimuths = 2048 if case["beams"] == 64 else 1090
    elevation = torch.linspace(-25.0, 3.0, case["beams"], device=device).mul(math.pi / 180)[:, None]
    turn = torch.rand(1, generator=gen, device=device) * (2 * math.pi / azimuths)
    azimuth = torch.arange(azimuths, device=device)[None] * (2 * math.pi / azimuths) + turn
    direction = torch.stack(torch.broadcast_tensors(elevation.cos() * azimuth.cos(),
                                                    elevation.cos() * azimuth.sin(), elevation.sin()), -1).reshape(-1, 3)
    origin = torch.tensor([at, 0.0, 1.8], device=device)
    ground = torch.where(direction[:, 2] < 0, -1.8 / direction[:, 2], torch.inf)
    t0, t1 = (low - origin) / direction[:, None], (high - origin) / direction[:, None]
    near, far = torch.minimum(t0, t1).amax(-1), torch.maximum(t0, t1).amin(-1)
    hit = torch.where((near <= far) & (near > 0), near, torch.inf).amin(1)
    distance = torch.minimum(ground, hit)
    distance = distance + 0.02 * torch.randn(distance.shape, generator=gen, device=device)
    return (origin + direction * distance[:, None])[(distance > 2) & (distance < 70)]


def _cells(case, points):
    """Voxel of every point, int64 [P, 3], not below zero, and which points are inside the range."""
    if case["kind"] == "detect":
        cell = torch.stack(((points[:, 2] + 3.2) / 0.2, (points[:, 1] + 54) / 0.075, (points[:, 0] + 54) / 0.075), 1)
        cell = cell.floor().long()
        return cell, ((cell >= 0) & (cell < torch.tensor(GRID, device=points.device))).all(1)
    low = torch.tensor([-75.0, -75.0, -0.5], device=points.device)
    return ((points - low) / case.get("voxel", 0.05)).floor().long(), torch.ones_like(points[:, 0], dtype=torch.bool)


def _cloud(case, gen, device):
    """float32 [P, 3] points of exactly case["voxels"] voxels, in the order they were measured:
    case["per_voxel"] of them per voxel on average where that is given."""
    want = case["voxels"]
    want_points = int(want * case.get("per_voxel", 1))
    scene, points = _scene(gen, device), torch.empty(0, 3, device=device)
    for sweep in range(400):
        points = torch.cat((points, _sweep(case, scene, 0.5 * sweep, gen, device)))
        cell, inside = _cells(case, points)
        points, cell = points[inside], cell[inside]
        key = (cell[:, 0] * 4096 + cell[:, 1]) * 4096 + cell[:, 2]
        voxels, of = torch.unique(key, return_inverse=True)
        if voxels.numel() < want:
            continue
        first = torch.full_like(voxels, points.shape[0]).scatter_reduce(
            0, of, torch.arange(points.shape[0], device=device), "amin")
        sector = torch.atan2(points[first, 1], points[first, 0] - 0.25 * sweep).argsort(stable=True)[:want]
        taken = torch.zeros_like(voxels, dtype=torch.bool)
        taken[sector] = True
        candidates = taken[of]
        if int(candidates.sum()) < want_points:
            continue
        keep = torch.zeros_like(candidates)
        keep[first[taken]] = True
        others = (candidates & ~keep).nonzero()[:, 0]
        if "per_voxel" in case:
            others = others[torch.randperm(others.numel(), generator=gen, device=device)[:want_points - want]]
        keep[others] = True
        return points[keep]
    raise RuntimeError("no such cloud: %r" % (case,))


def _clouds(case, seed, device):
    gen = torch.Generator(device=device).manual_seed(int(seed))
    return [_cloud(case, gen, device) for _ in range(case["scans"])]


def _voxels(case, clouds):
    """int32 [N, 4] (batch, x, y, z) voxels of the clouds in ascending order, as voxelisation by a ravelled
    key leaves them."""
    rows = []
    for b, points in enumerate(clouds):
        cell, _ = _cells(case, points)
        key = torch.unique((cell[:, 0] * 4096 + cell[:, 1]) * 4096 + cell[:, 2])
        cell = torch.stack((key >> 24, (key >> 12) & 4095, key & 4095), 1)
        if case["kind"] != "detect":
            cell -= cell.amin(0)
        rows.append(torch.cat((torch.full_like(cell[:, :1], b), cell), 1))
    return torch.cat(rows).int()


def _randn(shape, gen, dtype):
    return torch.randn(*shape, generator=gen, device="cuda").to(DTYPES[dtype])


# ------------------------------------------------------------------------------ preparation


def _network(case, net, x):
    """The network in the case's precision, its norms' statistics those of the given input."""
    norms = [m for m in net.modules() if isinstance(m, spnn.BatchNorm)]
    for m in norms:
        m.momentum = 1.0
    with torch.no_grad():
        net.train()(x)
    for m in norms:
        m.momentum = 0.1
    return net.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "loader":
        gen, clouds = torch.Generator(device="cuda").manual_seed(int(seed) + 1), []
        for cloud in _clouds(case, seed, "cuda"):
            at = _points_in_voxels(case, cloud, gen) * case["voxel"]
            clouds.append(torch.cat((at, torch.rand(len(at), 1, generator=gen, device="cuda")), 1).cpu().numpy())
        return {"case": case, "clouds": clouds}
    gen = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    torch.manual_seed(int(seed))
    if kind == "points":
        return _prepare_points(case, seed, gen)
    coords = _voxels(case, _clouds(case, seed, "cuda"))
    n = coords.shape[0]
    if kind == "maps":
        if case["shuffled"]:
            coords = coords[torch.randperm(n, generator=gen, device="cuda")].contiguous()
        return {"case": case, "coords": coords}
    state = {"case": case, "coords": coords}
    if kind == "layer":
        config = F.conv_config.get_default_conv_config()
        config.dataflow = DATAFLOWS[case["dataflow"]]
        layer = spnn.Conv3d(case["cin"], case["cout"], case["kernel"], stride=case["stride"],
                            padding=1 if case["kernel"] == 3 else 0, config=config).cuda().to(DTYPES[case["dtype"]])
        layer.train(case["backward"])
        x = ts.SparseTensor(_randn((n, case["cin"]), gen, case["dtype"]), coords)
        with torch.no_grad():
            rows = layer(x).feats.shape[0]  # (the maps are x's from here on)
        if case["backward"]:
            x.feats.requires_grad_()
            state["grad"] = _randn((rows, case["cout"]), gen, case["dtype"])
        return dict(state, layer=layer, x=x)
    channels = 5 if kind == "detect" else 4
    with torch.device("cuda"):
        net = (VoxelResBackBone8x if kind == "detect" else SparseResUNet42)(in_channels=channels)
        head = torch.nn.Linear(96, CLASSES).to(DTYPES[case["dtype"]])
    # position, and intensity (and time), standardised: what scans are given to networks with
    feats = torch.cat((coords[:, 1:].float(), torch.rand(n, channels - 3, generator=gen, device="cuda")), 1)
    feats = (feats - feats.mean(0)) / feats.std(0)
    state["range"] = (case["scans"],) + GRID if kind == "detect" else None
    net = _network(case, net, ts.SparseTensor(feats, coords, spatial_range=state["range"]))
    state["feats"] = feats.to(DTYPES[case["dtype"]])
    if kind == "train":
        state["labels"] = coords[:, 3].long() // 2 % CLASSES  # (something that can be learnt: height)
        params = list(net.parameters()) + list(head.parameters())
        state["sgd"] = torch.optim.SGD(params, lr=1e-8)
        state["kernels"] = [p for name, p in net.named_parameters() if name.endswith("kernel")]
    else:
        net = fuse_inference(net.eval())
    return dict(state, net=net, head=head)


def _points_in_voxels(case, cloud, gen):
    """float32 [P, 3] points of the cloud in units of its voxels, none closer to a border than rounding reaches."""
    cell, _ = _cells(case, cloud)
    return cell - cell.amin(0) + torch.rand(cloud.shape, generator=gen, device=cloud.device) * 0.98 + 0.01


def _prepare_points(case, seed, gen):
    """Points in voxel units with their batch index, and the voxels' coordinates and features."""
    clouds = _clouds(case, seed, "cuda")
    voxels, points = _voxels(case, clouds), []
    for b, cloud in enumerate(clouds):
        points.append(torch.cat((torch.full_like(cloud[:, :1], b), _points_in_voxels(case, cloud, gen)), 1))
    points = torch.cat(points)
    c = case["channels"]
    return {"case": case, "points": points, "voxels": voxels, "offsets": get_kernel_offsets(2, device="cuda"),
            "point_feats": _randn((points.shape[0], c), gen, case["dtype"]).requires_grad_(),
            "voxel_feats": _randn((voxels.shape[0], c), gen, case["dtype"]).requires_grad_(),
            "voxel_grad": _randn((voxels.shape[0], c), gen, case["dtype"]),
            "point_grad": _randn((points.shape[0], c), gen, case["dtype"])}


# ------------------------------------------------------------------------------ one pass


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _segment(state):
    with torch.no_grad():
        x = ts.SparseTensor(state["feats"], state["coords"].clone())  # (what a loader hands over: a new tensor)
        return state["head"](state["net"](x)[-1].feats)


def _train(state):
    net, head, sgd = state["net"], state["head"], state["sgd"]
    sgd.zero_grad(set_to_none=True)
    x = ts.SparseTensor(state["feats"], state["coords"].clone())
    scores = head(net(x)[-1].feats)
    loss = torch.nn.functional.cross_entropy(scores.float(), state["labels"])
    (loss * 1024).backward()  # (a static loss scale; the rate is small, so that many passes leave the network as it is)
    grads = [p.grad for p in state["kernels"]]
    # the norms of the gradients, which training programs watch and clip; their single values follow which
    # activations near zero are below it, and differ from one correct computation in 16 bits to the next
    norms = torch.stack(torch._foreach_norm([g.float() for g in grads]))
    sgd.step()
    return {"scores": scores.detach(), "loss": loss.detach(), "head_grad": head.weight.grad, "grad_norms": norms}


def _detect(state):
    with torch.no_grad():
        x = ts.SparseTensor(state["feats"], state["coords"].clone(), spatial_range=state["range"])
        return state["net"](x)["out"].dense()  # (the detector's head works on the dense bird's eye view)


def _layer(state):
    layer, x, case = state["layer"], state["x"], state["case"]
    # how many rows a strided layer has depends on the cloud; it has no fewer than these
    least = x.coords.shape[0] // case["stride"] ** 3
    if not case["backward"]:
        with torch.no_grad():
            return layer(x).feats[:least]
    x.feats.grad = layer.kernel.grad = None
    y = layer(x).feats
    y.backward(state["grad"])
    return y.detach()[:least], x.feats.grad, layer.kernel.grad


def _maps(state):
    case, coords = state["case"], state["coords"].clone()
    n, mode = coords.shape[0], "hashmap_on_the_fly"
    own = F.build_kernel_map(coords, n, case["kernel"], 1, 0, mode=mode)
    below = F.build_kernel_map(coords, n, case["down"], case["down"], 0, own["hashmap_keys"], own["hashmap_vals"],
                               mode=mode)
    rows, least = below["coords"].shape[0], n // case["down"] ** 3  # (there are no fewer rows than that)
    return own["out_in_map"][:n], rows, below["out_in_map"][:least], below["coords"][:least]


def _points(state):
    """Point-to-voxel and voxel-to-point as SPVCNN calls them, with their gradients."""
    points, voxels, point_feats, voxel_feats = (state[k] for k in ("points", "voxels", "point_feats", "voxel_feats"))
    point_feats.grad = voxel_feats.grad = None
    cells = points.floor().int()
    voxel_hash = F.sphash(voxels)
    index = F.sphashquery(F.sphash(cells), voxel_hash)
    counts = F.spcount(index, voxels.shape[0])
    means = F.spvoxelize(point_feats, index, counts)
    corners = F.sphashquery(F.sphash(cells, state["offsets"]), voxel_hash).t().contiguous()
    weights = F.calc_ti_weights(points[:, 1:], corners)
    values = F.spdevoxelize(voxel_feats, corners, weights)
    torch.autograd.backward((means, values), (state["voxel_grad"], state["point_grad"]))
    return {"index": index, "counts": counts, "weights": weights, "means": means.detach(),
            "values": values.detach(), "point_grad": point_feats.grad, "voxel_grad": voxel_feats.grad}


def _loader(state):
    samples, inverses = [], []
    for cloud in state["clouds"]:
        coords, index, inverse = sparse_quantize(cloud[:, :3], state["case"]["voxel"], return_index=True,
                                                 return_inverse=True)
        samples.append(ts.SparseTensor(torch.from_numpy(cloud[index]), torch.from_numpy(coords)))
        inverses.append(inverse)
    batch = sparse_collate(samples)
    return {"coords": batch.coords, "feats": batch.feats, "inverse": np.concatenate(inverses)}


_RUN = {"segment": _segment, "train": _train, "detect": _detect, "layer": _layer, "maps": _maps, "points": _points,
        "loader": _loader}

# ------------------------------------------------------------------------------ work and tolerance


def _packed(rows):
    b, x, y, z = (rows[:, i].astype(np.int64) + (0 if i == 0 else 8) for i in range(4))
    return ((b * 8192 + x) * 8192 + y) * 8192 + z


def _neighbours(rows, kernel):
    """Pairs of a submanifold map: (row, row) at most (kernel - 1) / 2 apart on every axis."""
    keys, half = np.sort(_packed(rows)), kernel // 2
    pairs = keys.size
    for d in range(kernel ** 3 // 2):  # (half of the offsets: the others mirror them)
        x, y, z = d // kernel ** 2 - half, d // kernel % kernel - half, d % kernel - half
        at = np.searchsorted(keys, keys + (x * 8192 + y) * 8192 + z)
        pairs += 2 * int((keys[np.minimum(at, keys.size - 1)] == keys + (x * 8192 + y) * 8192 + z).sum())
    return pairs


def _below(rows, kernel, stride, padding):
    """Output rows of a strided layer and the pairs of its map (3-tuples)."""
    outs = []
    for d in range(math.prod(kernel)):
        digit = np.array([d // (kernel[1] * kernel[2]), d // kernel[2] % kernel[1], d % kernel[2]])
        at = rows[:, 1:] + np.array(padding) - digit
        ok = (at % stride == 0).all(1) & (at >= 0).all(1)
        outs.append(np.concatenate((rows[ok, :1], at[ok] // stride), 1))
    outs = np.concatenate(outs)
    _, first = np.unique(_packed(outs), return_index=True)
    return outs[first], len(outs)


@lru_cache(maxsize=64)
def _geometry(items):
    """Rows and pairs of the maps a case builds, counted over clouds like its own.  Batches are one
    scan, times their number."""
    case = dict(items)
    times = case["scans"]
    rows = _voxels(case, _clouds(dict(case, scans=1), 0, "cpu")).numpy()
    levels, pairs, between = [len(rows)], [_neighbours(rows, case.get("kernel", 3) | 1)], []
    if case["kind"] == "layer" and case["stride"] > 1:
        pad = 1 if case["kernel"] == 3 else 0
        strides = [((case["kernel"],) * 3, (2, 2, 2), (pad,) * 3)]
    elif case["kind"] == "maps":
        strides = [((case["down"],) * 3, (case["down"],) * 3, (0, 0, 0))]
    elif case["kind"] == "detect":
        strides = [((3, 3, 3), (2, 2, 2), (1, 1, 1))] * 2 + [((3, 3, 3), (2, 2, 2), (0, 1, 1)),
                                                             ((3, 1, 1), (2, 1, 1), (0, 0, 0))]
    else:
        strides = [((2, 2, 2), (2, 2, 2), (0, 0, 0))] * 4 if case["kind"] in ("segment", "train") else []
    for kernel, stride, padding in strides:
        rows, between_pairs = _below(rows, kernel, stride, padding)
        levels.append(len(rows))
        pairs.append(_neighbours(rows, 3))
        between.append(between_pairs)
    return [times * v for v in levels], [times * v for v in pairs], [times * v for v in between]


def _network_layers(case):
    """(rows in, rows out, pairs, kernel volume, cin, cout) of every convolution of the network."""
    rows, pairs, between = _geometry(tuple(sorted(case.items())))
    layers = []

    def subm(level, cin, cout):
        layers.append((rows[level], rows[level], pairs[level], 27, cin, cout))

    if case["kind"] == "detect":
        subm(0, 5, 16)
        for level, c in enumerate((16, 32, 64, 128)):
            if level:
                layers.append((rows[level - 1], rows[level], between[level - 1], 27, c // 2, c))
            for _ in range(4):
                subm(level, c, c)
        layers.append((rows[3], rows[4], between[3], 3, 128, 128))
        return layers

    def block(level, cin, cout):
        subm(level, cin, cout)
        subm(level, cout, cout)
        if cin != cout:
            layers.append((rows[level], rows[level], rows[level], 1, cin, cout))

    skip = [32, 32, 64, 128, 256]
    subm(0, 4, 32)
    subm(0, 32, 32)
    for i in range(4):
        layers.append((rows[i], rows[i + 1], between[i], 8, skip[i], skip[i]))
        block(i + 1, skip[i], skip[i + 1])
        block(i + 1, skip[i + 1], skip[i + 1])
    c = 256
    for i, cout in enumerate((256, 128, 96, 96)):
        level = 3 - i
        layers.append((rows[level + 1], rows[level], between[level], 8, c, cout))
        block(level, cout + skip[level], cout)
        block(level, cout, cout)
        c = cout
    layers.append((rows[0], rows[0], rows[0], 1, 96, CLASSES))
    return layers


def work(case):
    """Bytes and operations of one pass.  Of a network: those of its convolutions, whose inputs and
    outputs exchange rows across the whole chip and so cross memory, three times over in training; the
    pairs of the maps are what is multiplied, and the maps are written once and read once."""
    kind = case["kind"]
    case = {k: v for k, v in case.items() if k != "name"}
    size = DTYPES[case["dtype"]].itemsize if "dtype" in case else 4
    if kind == "loader":
        voxels = case["scans"] * case["voxels"]
        points = voxels * case["per_voxel"]
        return {"bytes": points * (16 + 8) + voxels * (16 + 16), "flops": 0.0}  # cloud; inverse; rows and features
    if kind == "points":
        voxels, c = case["scans"] * case["voxels"], case["channels"]
        points = voxels * case["per_voxel"]
        # coordinates in; index, counts, corners, weights; each feature and gradient matrix once
        return {"bytes": points * (16 + 4 + 32 + 32 + 4 * c * size) + voxels * (16 + 4 + 4 * c * size),
                "flops": points * c * (2 + 2 + 2 * 16.0)}
    if kind == "maps":
        rows, pairs, between = _geometry(tuple(sorted(case.items())))
        return {"bytes": 32.0 * rows[0] + 4.0 * rows[0] * case["kernel"] ** 3 + rows[1] * (16 + 4 * case["down"] ** 3),
                "flops": 0.0}
    if kind == "layer":
        rows, pairs, between = _geometry(tuple(sorted(case.items())))
        strided = case["stride"] > 1
        n, m, nnz = rows[0], rows[1] if strided else rows[0], between[0] if strided else pairs[0]
        k, cin, cout = case["kernel"] ** 3, case["cin"], case["cout"]
        once = size * (n * cin + m * cout + k * cin * cout)
        return {"bytes": 4.0 * nnz + once * (2.0 if case["backward"] else 1.0),
                "flops": 2.0 * nnz * cin * cout * (3 if case["backward"] else 1)}
    layers, times = _network_layers(case), 3 if kind == "train" else 1
    rows, pairs, between = _geometry(tuple(sorted(case.items())))
    maps = 8.0 * (sum(pairs) + sum(between)) + 16.0 * sum(rows)
    return {"bytes": maps + times * size * sum(n * cin + m * cout + k * cin * cout for n, m, _, k, cin, cout in layers),
            "flops": times * 2.0 * sum(nnz * cin * cout for _, _, nnz, _, cin, cout in layers)}


def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype")
    if kind in ("maps", "loader"):
        return "exact"
    if kind == "points":  # indices and counts are whole numbers; means and values are 32-bit sums, rounded once
        return {"rel": {"fp16": 1e-3, "bf16": 8e-3, "fp32": 1e-5}[dtype]}
    if kind == "layer":  # one rounding of the result; the pair dataflows round the products as well
        return {"rel": {"fp16": 2e-3, "bf16": 1e-2, "fp32": 1e-5}[dtype]}
    if kind == "train":  # roundings of 49 layers and back, in the norms of gradients whose signs follow them
        return {"rel": {"fp16": 1.5e-2, "bf16": 4e-2, "fp32": 2e-4}[dtype]}
    # roundings of a network's layers one after the other
    return {"rel": {"fp16": 5e-3, "bf16": 3e-2, "fp32": 2e-5}[dtype]}
