"""The work a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public entry points: PointTransformerV3.forward (inference, encoder-only classification,
training with its backward), Point.serialization and voxelize.grid_sample. Sizes follow the baseline configurations
(rooms of about 100k voxels at 2 cm, 64-beam sweeps at 5 cm), the test-suite's small scenes, and what lies around them:
one small scan whose latency counts, a whole floor in one scene. Scans are synthetic, seeded, and keep the benchmark's
point density whatever their size.

    listed() -> cases      draw(rng) -> one more case of the same ranges
    prepare(case, seed) -> state      run(state) -> outputs of one pass
    work(case) -> {"bytes", "flops"}      tolerance(case)
"""
import functools
import math

import numpy as np
import torch

from pointtransformerv3_amd import Point, PointTransformerV3, ops, synthetic
from pointtransformerv3_amd.voxelize import grid_sample

DEVICE = "cuda:0"
ORDERS = ("z", "z-trans", "hilbert", "hilbert-trans")
HALF = {"fp16": torch.float16, "bf16": torch.bfloat16}
BENCH_ROOM_POINTS = 106_000   # points drawn per 8 x 6 x 3 m room in the benchmark batch (about 100k voxels of 2 cm)


def listed():
    return [
        # one small scan (an object on a table, a depth camera's frame thinned out): the user waits for this one answer
        dict(name="infer_fp16_scan_2k", kind="infer", dtype="fp16", scan="room", scenes=1, points=2_000, spread=0.0,
             overlap=False),
        # shape classification: a batch of small objects through the encoder alone
        dict(name="infer_fp16_cls_16x2k", kind="cls", dtype="fp16", scan="object", scenes=16, points=2_048, spread=0.3,
             overlap=False),
        # one LiDAR sweep as it comes off a vehicle, bf16 weights
        dict(name="infer_bf16_lidar_sweep", kind="infer", dtype="bf16", scan="lidar", scenes=1, points=86_000, spread=0.0,
             overlap=False),
        # one room, the ordinary single-scene inference
        dict(name="infer_fp16_room_100k", kind="infer", dtype="fp16", scan="room", scenes=1, points=100_800, spread=0.0,
             overlap=False),
        # the headline: four rooms per batch in a serving loop whose inputs are complete before each call
        dict(name="infer_fp16_rooms_4x100k", kind="infer", dtype="fp16", scan="room", scenes=4, points=100_800, spread=0.0,
             overlap=True),
        # a whole floor of a building as one scene: the largest inference
        dict(name="infer_fp16_floor_1m", kind="infer", dtype="fp16", scan="room", scenes=1, points=1_008_000, spread=0.0,
             overlap=False),
        # evaluation of a model kept in float, as the evaluators of a training framework call it
        dict(name="infer_fp32_room_100k", kind="infer", dtype="fp32", scan="room", scenes=1, points=100_800, spread=0.0,
             overlap=False),
        # validation inside a mixed-precision training run: float weights under autocast, ragged scenes
        dict(name="infer_amp_rooms_3x50k", kind="infer", dtype="amp", scan="room", scenes=3, points=50_400, spread=0.3,
             overlap=False),
        # a training step at the benchmark's batch, bf16 autocast: the largest case
        dict(name="train_bf16_rooms_4x100k", kind="train", dtype="bf16", scan="room", scenes=4, points=100_800, spread=0.0,
             overlap=False),
        # fine-tuning on small crops, fp16 autocast
        dict(name="train_fp16_crops_2x15k", kind="train", dtype="fp16", scan="room", scenes=2, points=15_000, spread=0.3,
             overlap=False),
        # curve codes, sort and inverse of a large batch: what a pipeline that stores serialized scans calls
        dict(name="serialize_8x150k", kind="serialize", dtype="int", scan="room", scenes=8, points=150_000, spread=0.3,
             overlap=False),
        # raw points to the batch the model takes
        dict(name="grid_sample_3x400k", kind="voxelize", dtype="fp32", scan="room", scenes=3, points=400_000, spread=0.3,
             overlap=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "infer", "cls", "train", "train", "serialize", "voxelize"])
    scan, spread, overlap = "room", round(rng.uniform(0.0, 0.4), 3), False
    if kind == "infer":
        dtype = rng.choice(["fp16", "fp16", "bf16", "fp32", "amp"])
        if dtype in HALF and rng.random() < 0.3:
            scan, scenes, points, spread = "lidar", rng.choice([1, 1, 2]), _log_uniform(rng, 20_000, 86_000), 0.0
        else:
            total = _log_uniform(rng, 2_000, 1_000_000 if dtype in HALF else 100_000)
            scenes = rng.choice([s for s in (1, 1, 2, 3, 4, 6) if total // s >= 1_000])
            points = total // scenes
        overlap = dtype in HALF and rng.random() < 0.3
    elif kind == "cls":
        dtype, scan = rng.choice(["fp16", "bf16"]), "object"
        scenes, points = rng.choice([1, 4, 13, 16, 32]), _log_uniform(rng, 1_024, 8_192)
    elif kind == "train":
        dtype = rng.choice(["fp16", "bf16"])
        total = _log_uniform(rng, 8_000, 400_000)
        scenes = rng.choice([s for s in (1, 2, 3, 4, 5) if total // s >= 2_000])
        points = total // scenes
    elif kind == "serialize":
        dtype, scenes, points = "int", rng.choice([1, 2, 5, 8]), _log_uniform(rng, 4_000, 150_000)
    else:
        dtype, scenes, points = "fp32", rng.choice([1, 2, 3]), _log_uniform(rng, 10_000, 400_000)
    return dict(kind=kind, dtype=dtype, scan=scan, scenes=scenes, points=points, spread=spread, overlap=overlap)


# ---- inputs -------------------------------------------------------------------------------------------------------

def _sizes(case):
    """Voxels of each scene: ragged by +-spread. They belong to the case: inputs of another seed have the same sizes."""
    rng = np.random.default_rng([case["scenes"], case["points"], int(1000 * case["spread"])])
    return [max(64, int(case["points"] * (1.0 + case["spread"] * (2.0 * rng.random() - 1.0)))) for _ in range(case["scenes"])]


def _room_points(n, rng):
    """A room (a floor, a crop) at the benchmark's density: the walls scale with the square root of the points."""
    return synthetic.room_points(n, rng.integers(2 ** 31)) * math.sqrt(n / BENCH_ROOM_POINTS)


def _object_points(n, rng):
    """The surface of an object in the unit ball: an ellipsoid with a box on it."""
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    p = d * rng.uniform(0.3, 0.8, size=3)
    on_box = rng.random(n) < 0.4
    cube = d / np.abs(d).max(1, keepdims=True) * rng.uniform(0.15, 0.5, size=3) + rng.uniform(-0.3, 0.3, size=3)
    return np.where(on_box[:, None], cube, p)


def _unique_voxels(pts, grid):
    """What synthetic.voxelize_unique keeps (the first point of every voxel, in input order), sorted on the GPU."""
    g = torch.from_numpy(np.floor((pts - pts.min(0)) / grid).astype(np.int32)).to(DEVICE)
    key = (g[:, 0].long() << 42) | (g[:, 1].long() << 21) | g[:, 2].long()
    key, at = torch.sort(key, stable=True)
    first = torch.ones_like(key, dtype=torch.bool)
    first[1:] = key[1:] != key[:-1]
    keep = torch.sort(at[first])[0]
    return g[keep].cpu().numpy(), keep.cpu().numpy()


def _scene(case, n, rng):
    """One scene of exactly n voxels, one point each: enough points are drawn, what is too much is left out."""
    more = 1.05
    while True:
        if case["scan"] == "lidar":
            # a sweep of 64 beams; the azimuth step follows from the voxels wanted (0.2 degrees: about 86k voxels)
            sc = synthetic.lidar_scene(rng.integers(2 ** 31), 0.05, az_step_deg=0.2 * 86_000 / (n * more))
            g, coord = sc["grid_coord"], sc["coord"]
        else:
            pts, grid = (_object_points, 0.01) if case["scan"] == "object" else (_room_points, 0.02)
            pts = pts(int(n * (more + 0.02)) + 32, rng)
            g, keep = _unique_voxels(pts, grid)
            coord = pts[keep].astype(np.float32)
        if len(g) >= n:
            keep = np.sort(rng.permutation(len(g))[:n])
            return dict(coord=coord[keep], grid_coord=g[keep])
        more *= 1.05


def _raw_scene(case, n, rng):
    """Raw points over exactly n occupied voxels of 2 cm, 1.3 points to a voxel, in random order."""
    g = _scene(case, n, rng)["grid_coord"].astype(np.float64)
    g -= g.min(0)
    hits = np.concatenate([np.arange(n), rng.integers(0, n, size=int(0.3 * n))])
    inside = 0.1 + 0.8 * rng.random((len(hits), 3))
    at = np.flatnonzero(~g.any(1))
    corner = int(at[0]) if len(at) else 0    # one point in the corner of the scene's bounding box
    g[corner] = 0.0
    inside[corner] = 0.0
    return ((g[hits] + inside) * 0.02)[rng.permutation(len(hits))].astype(np.float32)


@functools.lru_cache(maxsize=None)
def _model(kind, dtype, in_channels):
    """The model a program keeps (random-init weights): one per kind, weight type and input width."""
    torch.manual_seed(20)
    model = PointTransformerV3(in_channels=in_channels, cls_mode=kind == "cls")
    if kind == "train":
        return model.to(DEVICE).train()
    model = model.eval().requires_grad_(False)
    return model.to(HALF[dtype]).to(DEVICE) if dtype in HALF else model.to(DEVICE)


def _loss_gradient(grid_coord, dtype, gen):
    """What a 13-class linear head under a mean cross-entropy hands back to its (N, 64) input: labels that follow the
    place in the scene, the head's probabilities random; times a gradient scaler's factor in fp16."""
    n = len(grid_coord)
    head = torch.randn(13, 64, generator=gen, device=DEVICE) / 8
    at = grid_coord.float() / (grid_coord.max(0)[0].float() + 1.0)
    label = (at[:, 2] * 6).long() * 2 + (at[:, 0] * 2).long()
    d = torch.softmax(torch.randn(n, 13, generator=gen, device=DEVICE), 1)
    d[torch.arange(n, device=DEVICE), label] -= 1.0
    return d @ head * ((65536.0 if dtype == "fp16" else 1.0) / n)


def prepare(case, seed):
    rng = np.random.default_rng([int(seed), 7])
    sizes = _sizes(case)
    state = dict(kind=case["kind"], dtype=case["dtype"], seed=int(seed) % (2 ** 31))
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed) + 1)
    if case["kind"] == "voxelize":
        pts = [_raw_scene(case, n, rng) for n in sizes]
        coord = np.concatenate(pts)
        state["coord"] = torch.from_numpy(coord).to(DEVICE)
        state["offset"] = torch.from_numpy(np.cumsum([len(p) for p in pts])).to(DEVICE)
        state["feat"] = torch.rand(len(coord), 6, generator=gen, device=DEVICE)
        state["segment"] = torch.randint(0, 13, (len(coord),), generator=gen, device=DEVICE)
        return state
    d = synthetic.collate([_scene(case, n, rng) for n in sizes])
    state["grid_coord"] = torch.from_numpy(d["grid_coord"]).to(DEVICE)
    state["offset"] = torch.from_numpy(d["offset"]).to(DEVICE)
    if case["kind"] == "serialize":
        return state
    feat = (synthetic.lidar_features if case["scan"] == "lidar" else synthetic.room_features)(d["coord"], int(seed))
    feat = torch.from_numpy(feat).to(DEVICE)
    if case["scan"] == "lidar":
        feat[:, :3] /= 50.0   # metres to the range a network is fed with
    model = _model(case["kind"], case["dtype"] if case["kind"] != "train" else "fp32", feat.shape[1])
    state["model"], state["overlap"] = model, case["overlap"]
    if case["kind"] == "train":
        state["feat"] = feat
        state["dfeat"] = _loss_gradient(state["grid_coord"], case["dtype"], gen)
        state["params"] = list(model.parameters())
        norms = [m for m in model.modules() if isinstance(m, torch.nn.BatchNorm1d)]
        for m in norms:
            m.reset_running_stats()
        state["running"] = [b for m in norms for b in (m.running_mean, m.running_var)]
    else:
        state["feat"] = feat.to(HALF[case["dtype"]]) if case["dtype"] in HALF else feat
    return state


# ---- one pass -----------------------------------------------------------------------------------------------------

def _batch(state):
    return dict(feat=state["feat"], grid_coord=state["grid_coord"], offset=state["offset"])


def run(state):
    kind = state["kind"]
    if kind == "serialize":
        point = Point(grid_coord=state["grid_coord"], offset=state["offset"])
        point.serialization(order=ORDERS)
        return dict(code=point["serialized_code"], order=point["serialized_order"], inverse=point["serialized_inverse"])
    if kind == "voxelize":
        out = grid_sample(state["coord"], state["offset"], 0.02, feat=state["feat"], keys=(("segment", state["segment"]),))
        return {k: out[k] for k in ("coord", "grid_coord", "offset", "index", "inverse", "feat", "segment")}
    model = state["model"]
    torch.manual_seed(state["seed"])   # row shuffles of the orders, stochastic depth
    if kind == "train":
        for p in state["params"]:
            p.grad = None
        with torch.autocast("cuda", dtype=HALF[state["dtype"]]):
            feat = model(_batch(state))["feat"]
        feat.backward(state["dfeat"].to(feat.dtype))
        # gradients in one flat bucket, as a data-parallel step hands them on
        grads = torch.cat([p.grad.reshape(-1) for p in state["params"]])
        return dict(feat=feat.detach(), grads=grads, running=torch.cat(state["running"]))
    model.overlap_index_prologue = state["overlap"]
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16, enabled=state["dtype"] == "amp"):
        point = model(_batch(state))
    if kind == "cls":
        # one descriptor per object: the mean over its pooled points
        ends = torch.nn.functional.pad(point["offset"], (1, 0))
        rows = torch.arange(point["feat"].shape[0], device=DEVICE)
        return dict(feat=ops.segment_reduce(point["feat"], rows, ends, "mean"))
    return dict(feat=point["feat"])


# ---- what a pass cannot do without --------------------------------------------------------------------------------

# points of a level over the points of level 0, and pairs of the 3x3x3 convolution per voxel, on the benchmark batch
LEVEL_SHARE = (1.0, 0.766, 0.363, 0.0935, 0.0214)
LEVEL_PAIRS = (2.46, 5.34, 9.73, 11.4, 12.6)
ENC = ((2, 32), (2, 64), (2, 128), (6, 256), (2, 512))
DEC = ((2, 64), (2, 64), (2, 128), (2, 256))
PARAMS = 46.2e6
PARAMS_ENCODER = 38.7e6


def _forward_flops(n, scenes, decoder):
    total = 2.0 * 5.0 * n * 6 * 32   # the stem: about five of its 125 taps are occupied
    stages = list(zip(ENC, LEVEL_SHARE, LEVEL_PAIRS)) + (list(zip(DEC, LEVEL_SHARE, LEVEL_PAIRS)) if decoder else [])
    for (depth, c), share, pairs in stages:
        rows = max(n * share, 1.0)
        patch = min(1024.0, max(1.0, rows / scenes))
        total += depth * rows * (2.0 * pairs * c * c + 2.0 * 13.0 * c * c + 4.0 * patch * c)
    for lo in range(4):
        c_in, c_out = ENC[lo][1], ENC[lo + 1][1]
        total += 2.0 * n * LEVEL_SHARE[lo] * c_in * c_out
        if decoder:
            below = DEC[lo + 1][1] if lo < 3 else ENC[4][1]
            total += 2.0 * n * (LEVEL_SHARE[lo] * ENC[lo][1] + LEVEL_SHARE[lo + 1] * below) * DEC[lo][1]
    return total


def work(case):
    n = float(case["scenes"] * case["points"])
    if case["kind"] == "serialize":
        return dict(bytes=n * (12.0 + 3 * 8.0 * len(ORDERS)), flops=0.0)
    if case["kind"] == "voxelize":
        # coordinates of every raw point in, its voxel out; the kept points' rows (coordinates, features, label) in and
        # out, their grid coordinates and index out
        return dict(bytes=n * (1.3 * (12.0 + 8.0) + 2 * (24.0 + 8.0) + 12.0 + 12.0 + 8.0), flops=0.0)
    decoder = case["kind"] != "cls"
    flops = _forward_flops(n, case["scenes"], decoder)
    width = 2.0 if case["dtype"] in HALF and case["kind"] != "train" else 4.0
    c_in = 4.0 if case["scan"] == "lidar" else 6.0
    rows_out = n * 64.0 if decoder else case["scenes"] * 512.0
    byts = n * (12.0 + c_in * width) + (PARAMS if decoder else PARAMS_ENCODER) * width + rows_out * width
    if case["kind"] == "train":
        flops *= 3.0
        byts += PARAMS * 4.0 + n * 64.0 * 4.0
    return dict(bytes=byts, flops=flops)


def tolerance(case):
    if case["kind"] in ("serialize", "voxelize"):
        return "exact"
    if case["kind"] == "train":
        # gradients of a whole network whose activations are rounded to 16 bits at every layer
        return dict(rel=0.03, max=0.99)
    if case["dtype"] == "fp32":
        return dict(rel=2e-3)   # the patch attention of a float model reads q, k and v in half precision
    return dict(rel=2.5e-2 if case["dtype"] == "bf16" else 1e-2)
