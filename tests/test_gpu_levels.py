"""The batched index pass against the separate per-level operators, table by table."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, to_dev, unique_voxels

pytestmark = pytest.mark.gpu


def _scenes(seed, sizes, extent):
    rng = np.random.default_rng(seed)
    grids, ends = [], []
    for n in sizes:
        if n:
            grids.append(unique_voxels(rng, n, extent)[0])
        ends.append(n)
    return np.concatenate(grids), np.cumsum(ends).astype(np.int64)


@pytest.mark.parametrize("sizes,extent,orders,patch,strides,only128", [
    ([1], 4, ("z", "hilbert"), 16, (2, 2), False),
    ([700], 40, ("z", "z-trans", "hilbert", "hilbert-trans"), 64, (2, 2, 2, 2), False),
    ([300, 0, 5, 1000], 30, ("z", "z-trans", "hilbert", "hilbert-trans"), 48, (2, 2, 2, 2), True),
    ([256, 255], 9, ("hilbert",), 100, (4,), False),
    ([5000, 9000], 1500, ("z", "z-trans", "hilbert", "hilbert-trans"), 1024, (2, 2, 2, 2), True),     # 33 and more key bits
    ([20000, 33000], 60, ("hilbert", "z"), 128, (2, 8, 2), False),
    ([4096, 1], 17, ("z",), 32, (), False),
])
def test_index_pass_equals_separate_operators(sizes, extent, orders, patch, strides, only128):
    from pointtransformerv3_amd import levels as L
    from pointtransformerv3_amd import ops
    grid_np, ends = _scenes(sum(sizes), sizes, extent)
    grid, offset = to_dev(grid_np), to_dev(ends)
    nb, k, n_levels = len(ends), len(orders), len(strides) + 1
    convs = [[(128, 128)] if only128 else [(64, 64)]] * n_levels
    layout = L.Layout(k, strides, [patch] * n_levels, [range(k)] * n_levels, convs, True, [True] * len(strides), only_pads0=False)
    torch.manual_seed(5)
    idx = L.build(layout, grid, offset, None, list(orders), True, lambda lv, level: L.PAIRS | L.TILES | L.PAIRS5)
    # the same through the separate operators
    torch.manual_seed(5)
    n = len(grid_np)
    batch = ops.offset2batch(offset, n)
    depth = int(grid_np.max()).bit_length()
    perm = torch.randperm(k).tolist()
    perms = [torch.randperm(k).tolist() for _ in strides]
    code = ops.encode_orders(grid, batch, depth, [orders[i] for i in perm])
    order, inverse = ops.argsort_rows(code, 3 * depth + max(1, (nb - 1).bit_length()))
    assert torch.equal(idx.batch, batch) and torch.equal(idx.code, code)
    assert torch.equal(idx.order, order) and torch.equal(idx.inverse, inverse)
    cur = dict(grid=grid, batch=batch, code=code, order=order, inverse=inverse, offset=offset, host=[int(v) for v in ends])
    indices = torch.cat([batch[:, None].int(), grid], 1).contiguous()
    i64, i32 = torch.int64, torch.int32
    for lv in range(n_levels):
        v = idx.levels[lv]
        if lv:
            d = (int(np.ceil(strides[lv - 1])) - 1).bit_length()
            d = 0 if d > depth else d
            depth -= d
            cluster, idx_ptr, head, m, off, host = ops.pool_clusters(cur["code"][0], cur["order"][0], 3 * d, cur["offset"])
            p = perms[lv - 1]
            c2, g2, b2, indices = ops.pool_gather(cur["code"], 3 * d, cur["grid"], d, cur["batch"], head, p)
            o2, i2 = ops.pool_orders(cur["order"], cluster, m, p)
            assert v.n == m and v.depth == depth
            got = lambda ptr, shape, dt: idx.tensor(ptr, shape, dt)
            assert torch.equal(got(v.code, (k, m), i64), c2)
            assert torch.equal(got(v.order, (k, m), i64), o2)
            assert torch.equal(got(v.inverse, (k, m), i64), i2)
            assert torch.equal(got(v.grid, (m, 3), i32), g2)
            assert torch.equal(got(v.batch, (m,), i64), b2)
            assert torch.equal(got(v.indices, (m, 4), i32), indices)
            assert torch.equal(got(v.cluster, (len(cluster),), i64), cluster)
            assert torch.equal(got(v.idx_ptr, (m + 1,), i64), idx_ptr)
            assert torch.equal(idx.tensor(v.offset, (nb,), i64, "first"), off)
            assert idx.level_offsets[lv] == host
            cur = dict(grid=g2, batch=b2, code=c2, order=o2, inverse=i2, offset=off, host=host)
        m = v.n
        pad, unpad, cu = ops.pad_index(cur["offset"], cur["host"], patch)
        assert torch.equal(idx.tensor(v.pad, (v.n_pad,), i64), pad)
        assert torch.equal(idx.tensor(v.unpad, (m,), i64), unpad)
        assert torch.equal(idx.tensor(v.cu, (v.n_seq + 1,), i32), cu)
        for r in range(k):
            src, dst = ops.attn_slots(cur["order"][r], cur["inverse"][r], pad, unpad)
            assert torch.equal(idx.tensor(v.slot_src[r], (v.n_pad,), i32), src)
            assert torch.equal(idx.tensor(v.slot_dst[r], (v.n_pad,), i32), dst)
        for ks in ((3, 5) if lv == 0 else (3,)):
            plan = ops.conv_plan_direct(indices, ks)
            s = "5" if ks == 5 else ""
            pairs = getattr(v, "n_pairs" + s)
            assert pairs == plan.n_pairs
            where = "first" if lv == 0 else "scratch"
            assert torch.equal(idx.tensor(getattr(v, "tap_ptr" + s), (ks ** 3 + 1,), i32, where), plan.tap_ptr)
            assert torch.equal(idx.tensor(getattr(v, "row_ptr" + s), (m + 1,), i32, "lists"), plan.row_ptr)
            assert torch.equal(idx.tensor(getattr(v, "pair_in" + s), (pairs,), i32, "lists"), plan.pair_in[:pairs])
            assert torch.equal(idx.tensor(getattr(v, "pair_slot" + s), (pairs,), i32, "lists"), plan.pair_slot[:pairs])
            if ks == 3:
                tv = ops.tile_voxels_for(m, 128) if only128 else 128
                assert v.tile_voxels == tv
                tile_tap, tile_pair, vox_taps = plan.tiles(tv)
                assert torch.equal(idx.tensor(v.tile_tap, tuple(tile_tap.shape), i32, "lists"), tile_tap)
                assert torch.equal(idx.tensor(v.tile_pair, (pairs,), i32, "lists"), tile_pair[:pairs])
                assert torch.equal(idx.tensor(v.vox_taps, (m,), i32, "lists"), vox_taps)
                only = L.build(layout, grid, offset, None, list(orders), False, lambda lv, level: L.TILES).levels[lv]
                assert only.n_pairs == pairs


@pytest.mark.parametrize("want", [1, 2])
def test_index_pass_single_list_kinds(want):
    """Pairs alone and tiles alone are the lists that both together give."""
    from pointtransformerv3_amd import levels as L
    grid_np, ends = _scenes(3, [900, 2500], 25)
    grid, offset = to_dev(grid_np), to_dev(ends)
    layout = L.Layout(2, (2, 2), [64] * 3, [range(2)] * 3, [[(64, 64)]] * 3, False, [False, False])
    both = L.build(layout, grid, offset, None, ["z", "hilbert"], False, lambda lv, level: L.PAIRS | L.TILES)
    one = L.build(layout, grid, offset, None, ["z", "hilbert"], False, lambda lv, level: want)
    fields = [("row_ptr", 1), ("pair_in", 0), ("pair_slot", 0)] if want == 1 else [("tile_pair", 0), ("vox_taps", 2)]
    for lv in range(3):
        for f, kind in fields:
            m, p = both.levels[lv].n, both.levels[lv].n_pairs
            shape = ((p,), (m + 1,), (m,))[kind]
            assert torch.equal(both.tensor(getattr(both.levels[lv], f), shape, torch.int32, "lists"),
                               one.tensor(getattr(one.levels[lv], f), shape, torch.int32, "lists"))


@pytest.mark.parametrize("train", [False, True])
def test_nothing_of_the_index_scratch_outlives_the_index(train):
    """Bytes that stay allocated for a forward's result: its own tensors and the tables its keys are views of (about 100
    bytes a point of codes, orders and inverses, up to 300 of pooled tables), no voxel hash."""
    from pointtransformerv3_amd import PointTransformerV3, synthetic
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0).to(DEV)
    model = model.train() if train else model.eval().half()
    d = synthetic.collate([synthetic.room_scene(60_000, 5 + i, 0.02) for i in range(2)])
    data = dict(feat=torch.from_numpy(synthetic.room_features(d["coord"], 1)).to(DEV).to(torch.float32 if train else torch.float16),
                grid_coord=torch.from_numpy(d["grid_coord"]).to(DEV), offset=torch.from_numpy(d["offset"]).to(DEV))
    n = data["feat"].shape[0]

    def forward():
        if train:
            with torch.autocast("cuda", dtype=torch.bfloat16):
                return model(dict(data))
        with torch.inference_mode():
            return model(dict(data))

    forward()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    point = forward()
    if train:
        point.feat.sum().backward()
        grads = sum(p.numel() * 4 for p in model.parameters())
        point.feat = point.feat.detach()
        point.sparse_conv_feat.features = point.feat
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated() - before - (grads if train else 0)
    indices = point.sparse_conv_feat.indices
    assert indices.untyped_storage().nbytes() <= 16 * n + 4096
    assert held <= n * (16 + 96 + 8 + 64 * point.feat.element_size() + 330) + (1 << 20), held / n
