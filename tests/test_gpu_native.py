"""The natively queued inference forward against the same model's modules."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import DEV, rel_err

pytestmark = pytest.mark.gpu

KW = dict(enc_depths=(1, 1, 2, 1, 1), dec_depths=(1, 2, 1, 1), enc_patch_size=(256,) * 5, dec_patch_size=(256,) * 4)


def _inputs(seed, sizes, dtype, grid=0.04):
    from pointtransformerv3_amd import synthetic
    d = synthetic.collate([synthetic.room_scene(n, seed + i, grid) for i, n in enumerate(sizes)])
    feat = torch.from_numpy(synthetic.room_features(d["coord"], seed)).to(DEV).to(dtype)
    return dict(feat=feat, coord=torch.from_numpy(d["coord"]).to(DEV), grid_coord=torch.from_numpy(d["grid_coord"]).to(DEV),
                offset=torch.from_numpy(d["offset"]).to(DEV))


def _both(model, data, monkeypatch, amp=None):
    from pointtransformerv3_amd import native
    taken, real = [], native.engine_for
    outs = []
    for use in (True, False):
        monkeypatch.setattr(native, "engine_for",
                            (lambda m, d: taken.append(real(m, d)) or taken[-1]) if use else (lambda m, d: None))
        torch.manual_seed(9)
        with torch.inference_mode(), torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            outs.append(model(dict(data)))
    monkeypatch.setattr(native, "engine_for", real)
    assert taken[0] is not None, "the native path was not taken"
    return outs


@pytest.mark.parametrize("sizes", [(5000,), (9000, 61, 4000), (40,)])
@pytest.mark.parametrize("dtype,amp", [(torch.float16, None), (torch.bfloat16, None), (torch.float32, None),
                                       (torch.float32, torch.float16)])
def test_native_forward_equals_the_modules(dtype, amp, sizes, monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().to(dtype).to(DEV)
    got, want = _both(model, _inputs(4, sizes, dtype), monkeypatch, amp)
    assert got.feat.dtype == want.feat.dtype
    assert torch.equal(got.feat, want.feat)
    for key in ("batch", "offset", "serialized_code", "serialized_order", "serialized_inverse", "pad", "unpad", "cu_seqlens_key"):
        assert torch.equal(got[key], want[key]), key
    assert got.serialized_depth == want.serialized_depth and got.sparse_shape == want.sparse_shape
    assert torch.equal(got.sparse_conv_feat.indices, want.sparse_conv_feat.indices)
    assert torch.equal(got.sparse_conv_feat.features, want.feat)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_native_forward_with_weights_asked_for_ahead(dtype, monkeypatch):
    """A level of 256 channels beyond the layers of few rows: the attention and the convolution's sum ask for the next kernel's
    weights, which the modules' launches do not."""
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().to(dtype).to(DEV)
    got, want = _both(model, _inputs(4, (40_000,), dtype, grid=0.02), monkeypatch)
    assert got.feat.shape[0] > 30_000 and torch.equal(got.feat, want.feat)


def test_native_forward_without_the_packed_first_half_at_256_channels():
    """A description without that copy takes the separate layers, as descriptions did before there was one: the same roundings,
    sums in another order."""
    from pointtransformerv3_amd import PointTransformerV3, native
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().half().to(DEV)
    data = _inputs(4, (40_000,), torch.float16, grid=0.02)
    outs = []
    with torch.inference_mode():
        for drop in (False, True):
            torch.manual_seed(9)
            outs.append(model(dict(data)).feat.float())
            engine = native.engine_for(model, data)
            left_out = [b for a in engine._keep if isinstance(a, ctypes.Array) and a._type_ is native._Block for b in a if b.channels == 256]
            assert left_out and all(bool(b.head_packed) != drop for b in left_out)
            for b in left_out:
                b.head_packed = None
    assert rel_err(outs[1], outs[0].cpu()) < 2e-2


@pytest.mark.parametrize("reduce,stride,sizes", [("max", (2, 2, 2, 2), (5003, 61)), ("mean", (8, 2, 2, 2), (9000,)), ("min", (2, 2, 2, 2), (40,)),
                                                ("sum", (4, 2, 2, 2), (3000, 500))])
@pytest.mark.parametrize("dtype,stats", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                                         (torch.float16, torch.float32)])
def test_norms_behind_a_reduction_equal_the_modules(dtype, stats, reduce, stride, sizes, monkeypatch):
    """Statistics, scales and shifts of their own, short and long segments: the bits of the separate passes."""
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(stride=stride, cls_mode=True, **KW).eval().to(dtype).to(DEV)
    for m in model.modules():
        if type(m).__name__ == "BatchNorm1d":
            m.running_mean = torch.randn_like(m.running_mean).to(stats) * 0.3
            m.running_var = torch.rand_like(m.running_var).to(stats) + 0.2
            m.weight.data.uniform_(-1.5, 1.5)
            m.bias.data.uniform_(-0.5, 0.5)
        if type(m).__name__ == "SerializedPooling":
            m.reduce = reduce
    got, want = _both(model, _inputs(4, sizes, dtype), monkeypatch)
    assert torch.isfinite(want.feat).all() and torch.equal(got.feat, want.feat)


def test_native_encoder_only_fills_every_level(monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(cls_mode=True, **KW).eval().half().to(DEV)
    got, want = _both(model, _inputs(4, (3000, 7000), torch.float16), monkeypatch)
    depth = 0
    while True:
        keys = {k for k in want if isinstance(want[k], torch.Tensor) and not k.startswith("_")}
        assert keys <= set(got) and got.serialized_depth == want.serialized_depth
        for key in keys:
            assert torch.equal(got[key], want[key]), (depth, key)
        if "pooling_parent" not in want:
            break
        got, want, depth = got.pooling_parent, want.pooling_parent, depth + 1
    assert depth == 4


def test_native_forward_follows_changed_weights_and_leaves_changed_models_alone(monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3, native
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().half().to(DEV)
    data = _inputs(7, (4000,), torch.float16)
    first = _both(model, data, monkeypatch)[0].feat
    model.enc.enc2.block0.mlp[0].fc1.weight.data.mul_(1.5)                     # in place, behind autograd's back
    got, want = _both(model, data, monkeypatch)
    assert torch.equal(got.feat, want.feat) and not torch.equal(got.feat, first)
    model.dec.dec1.block0.attn.qkv.weight = torch.nn.Parameter(model.dec.dec1.block0.attn.qkv.weight.data * 0.5)   # another tensor
    got, want = _both(model, data, monkeypatch)
    assert torch.equal(got.feat, want.feat)
    with torch.inference_mode():
        handle = model.enc.enc1.register_forward_hook(lambda m, a, r: None)    # hooks want the modules to run
        assert native.engine_for(model, data) is None
        handle.remove()
        assert native.engine_for(model, data) is not None
        assert native.engine_for(model, dict(data, sparse_shape=[1, 2, 3])) is None
        model.enc.enc1.down.norm[0].train()
        assert native.engine_for(model, data) is None
        model.eval()
        model.dec.dec0.block0.mlp[0].fc1 = torch.nn.Sequential(model.dec.dec0.block0.mlp[0].fc1)   # not the default architecture
        assert native.engine_for(model, data) is None
    assert native.engine_for(model, data) is None                              # grad mode: the modules


def _each(model, kind, name, value):
    for m in model.modules():
        if type(m).__name__ == kind:
            setattr(m, name, value)


@pytest.mark.parametrize("change,native_again", [
    (lambda m: _each(m, "LayerNorm", "eps", 1e-2), True), (lambda m: _each(m, "BatchNorm1d", "eps", 0.5), True),
    (lambda m: _each(m, "SerializedAttention", "scale", 0.6), True), (lambda m: _each(m, "SerializedAttention", "patch_size", 64), True),
    (lambda m: _each(m, "SerializedAttention", "order_index", 1), True),
    (lambda m: _each(m, "SerializedPooling", "reduce", "mean"), True),
    (lambda m: _each(m, "SerializedPooling", "shuffle_orders", False), True),
    (lambda m: _each(m, "GELU", "approximate", "tanh"), False),
    (lambda m: m.enc.enc1.add(torch.nn.LayerNorm(64).half().to(DEV), name="extra"), False),
    (lambda m: setattr(m.enc.enc2.block0.mlp[0], "forward", lambda x: x), False),
    (lambda m: m.dec.dec0._modules.pop("block0"), True), (lambda m: setattr(m.enc.enc2.block0.mlp[0].fc1, "bias", None), False)],
    ids=["layer_norm_eps", "batch_norm_eps", "scale", "patch_size", "order_index", "reduce", "shuffle_orders", "gelu", "child_added",
         "forward", "child_removed", "no_bias"])
def test_a_model_changed_after_its_first_forward_is_described_again_or_left_to_the_modules(change, native_again, monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3, native
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().half().to(DEV)
    data = _inputs(7, (4000, 900), torch.float16)
    _both(model, data, monkeypatch)
    change(model)
    real = native.engine_for
    outs = []
    for use in (True, False):
        taken = []
        monkeypatch.setattr(native, "engine_for", (lambda m, d: taken.append(real(m, d)) or taken[-1]) if use else (lambda m, d: None))
        torch.manual_seed(9)
        with torch.inference_mode():
            try:
                outs.append(model(dict(data)).feat)
            except Exception as e:      # what the modules refuse is refused the same way
                outs.append(type(e))
        if use:
            assert (taken[0] is not None) == native_again
    got, want = outs
    assert type(got) is type(want) and (torch.equal(got, want) if isinstance(want, torch.Tensor) else got is want)


def test_models_that_ran_are_freed(monkeypatch):
    """A model's weights and the copies made of them go with the model, in evaluation and training."""
    import gc
    from pointtransformerv3_amd import PointTransformerV3
    data = _inputs(7, (2000,), torch.float16)

    def run(train):
        model = PointTransformerV3(**KW).to(DEV)
        if train:
            model.train()
            with torch.autocast("cuda", dtype=torch.float16):
                model(dict(data, feat=data["feat"].float())).feat.sum().backward()
        else:
            with torch.inference_mode():
                model.eval().half()(dict(data))
        del model
        gc.collect()
        torch.cuda.synchronize()
        return torch.cuda.memory_allocated()

    for train in (False, True):
        held = [run(train) for _ in range(3)]
        assert held[2] == held[1], held          # the first run may leave fixed workspaces behind


@pytest.mark.parametrize("train", [False, True])
def test_copies_outlive_their_engine_where_another_stream_reads_them(train):
    """A model that is described again, or deleted, while a forward on a second stream still runs."""
    from pointtransformerv3_amd import PointTransformerV3, native, native_train
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV)
    model = model.train() if train else model.eval().half()
    data = _inputs(7, (2000,), torch.float32 if train else torch.float16)
    side = torch.cuda.Stream()

    def run():
        if train:
            with torch.autocast("cuda", dtype=torch.float16):
                return model(dict(data)).feat
        with torch.inference_mode():
            return model(dict(data)).feat

    run()
    engine = next(iter((native_train if train else native)._ENGINES[model].values()))
    copies = [t for t in engine._keep if isinstance(t, torch.Tensor)]
    marked = []
    torch.cuda.synchronize()
    real = torch.Tensor.record_stream
    torch.Tensor.record_stream = lambda t, s: marked.append((t.data_ptr(), s.cuda_stream)) or real(t, s)
    try:
        with torch.cuda.stream(side):
            run()
            run()
    finally:
        torch.Tensor.record_stream = real
    torch.cuda.synchronize()
    wanted = [(t.data_ptr(), side.cuda_stream) for t in copies]
    assert [m for m in marked if m in wanted] == wanted      # each of them, once


def _volume(extent, dtype, fill=1.0):
    """A solid block of voxels: most taps of most voxels are there."""
    g = np.stack(np.meshgrid(*[np.arange(extent)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[np.random.default_rng(extent).random(len(g)) < fill].astype(np.int32)
    gen = torch.Generator(device=DEV).manual_seed(extent)
    return dict(feat=torch.randn(len(g), 6, generator=gen, device=DEV).to(dtype), grid_coord=torch.from_numpy(g).to(DEV),
                offset=torch.tensor([len(g)], device=DEV))


@pytest.mark.parametrize("extent,fill", [(12, 1.0), (32, 1.0), (32, 0.8)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_native_forward_takes_the_modules_forms_in_dense_volumes(dtype, extent, fill, monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3, ops
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().to(dtype).to(DEV)
    dense, real = [], ops.subm_conv
    monkeypatch.setattr(ops, "subm_conv", lambda x, *a, **k: dense.append(x.shape) or real(x, *a, **k))
    got, want = _both(model, _volume(extent, dtype, fill), monkeypatch)
    assert torch.equal(got.feat, want.feat)
    assert bool(dense) == (dtype == torch.float16 and extent == 32)


def test_dense_volumes_follow_the_module_class_setting(monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3, SubMConv3d
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().half().to(DEV)
    data = _volume(32, torch.float16)
    first = _both(model, data, monkeypatch)[0].feat
    monkeypatch.setattr(SubMConv3d, "PAIR_MODE_MAX_DENSITY", 1.0)
    got, want = _both(model, data, monkeypatch)
    assert torch.equal(got.feat, want.feat) and not torch.equal(got.feat, first)


def test_one_model_in_several_threads_and_streams():
    """Threads with a stream of their own each run one model on different inputs: the results of one after the other."""
    import threading
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(shuffle_orders=False, **KW).eval().to(DEV)
    _each(model, "SerializedPooling", "shuffle_orders", False)
    datas = [_inputs(s, sizes, torch.float32) for s, sizes in ((4, (5000,)), (11, (3000, 700)), (23, (9000,)), (31, (2500, 2500)))]
    torch.cuda.synchronize()

    def run(data):
        with torch.inference_mode(), torch.autocast("cuda", dtype=torch.float16):     # weight copies made by every forward
            return model(dict(data)).feat

    want = [run(d) for d in datas]
    torch.cuda.synchronize()
    got, failed = [[] for _ in datas], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(6):
                    got[i].append(run(datas[i]))
                torch.cuda.current_stream().synchronize()
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(datas))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed and not any(t.is_alive() for t in threads)
    for w, rows in zip(want, got):
        assert len(rows) == 6 and all(torch.equal(w, r) for r in rows)


def test_inputs_that_kernels_cannot_address_are_not_taken():
    """Other shapes and places than the kernels assume go to the modules; scene ends that are none are refused before any
    table is made from them."""
    from pointtransformerv3_amd import PointTransformerV3, native
    from pointtransformerv3_amd._lib import Ptv3Error
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).eval().half().to(DEV)
    data = _inputs(7, (1500, 900), torch.float16)
    n = data["feat"].shape[0]
    batch = torch.zeros(n, dtype=torch.int64, device=DEV)
    batch[int(data["offset"][0]):] = 1
    with torch.inference_mode():
        want = model(dict(data)).feat
        assert native.engine_for(model, dict(data, batch=batch)) is not None
        for change in (dict(grid_coord=data["grid_coord"].cpu()), dict(offset=data["offset"].cpu()), dict(batch=batch.cpu()),
                       dict(batch=batch[:-1]), dict(batch=batch[:, None]), dict(offset=data["offset"][:, None]),
                       dict(grid_coord=torch.cat([data["grid_coord"]] * 2, 1)), dict(grid_coord=data["grid_coord"][:-1]),
                       dict(offset=data["offset"].tolist()), dict(offset=data["offset"][:0])):
            assert native.engine_for(model, dict(data, **change)) is None, list(change)
        without = {k: v for k, v in data.items() if k != "grid_coord"}
        assert native.engine_for(model, without) is None                     # coordinates, but no grid size
        assert native.engine_for(model, dict(without, grid_size=0.04)) is not None
        for ends in ([n - 1], [n + 1], [n + 5, n], [n, 5, n]):
            with pytest.raises(Ptv3Error):
                model(dict(data, offset=torch.tensor(ends, device=DEV)))
        assert torch.equal(model(dict(data, offset=torch.tensor([0, int(data["offset"][0]), n], device=DEV))).offset,
                           torch.tensor([0, int(data["offset"][0]), n], device=DEV))   # an empty scene is one
        torch.manual_seed(9)
        a = model(dict(data, batch=batch)).feat
        torch.manual_seed(9)
        assert torch.equal(a, model(dict(data)).feat) and want.shape == a.shape
