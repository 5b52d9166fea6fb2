"""Host-side rules of the natively queued paths that need no GPU."""
import contextlib
import ctypes
import gc
import types
import weakref

import pytest
import torch

from pointtransformerv3_amd import native, native_train


class _Stop(Exception):
    pass


@pytest.mark.parametrize("overlap", [True, False])
def test_inputs_are_converted_where_the_index_reads_them(overlap, monkeypatch):
    """Under the overlapped schedule the index stream waits for nothing: a conversion queued on the caller's stream would
    still be pending when the index kernels read its result."""
    inside, seen = [False], []

    class Overlap:
        device = torch.device("cpu")

        @contextlib.contextmanager
        def scope(self):
            inside[0] = True
            yield
            inside[0] = False

    def build(*args, **kw):
        raise _Stop

    monkeypatch.setattr(native.ops, "_stream", lambda: None)
    monkeypatch.setattr(native, "coordinates", lambda point: seen.append(inside[0]) or (None, None, None))
    monkeypatch.setattr(native.levels, "build", build)
    engine = native.Engine.__new__(native.Engine)
    engine.layout = engine.want = None
    engine.used_here = lambda: None
    engine._refresh = native._Refresh()   # nothing to refresh: launches nothing
    model = types.SimpleNamespace(overlap_index_prologue=overlap, _prologue_state=Overlap(), order=("z",), shuffle_orders=False)
    with pytest.raises(_Stop):
        engine.forward(model, dict(feat=torch.zeros(4, 6), grid_coord=torch.zeros(4, 3, dtype=torch.int64), offset=torch.tensor([4])))
    assert seen == [overlap]


class _TrainLib:
    """Stands in for the library: the two calls of a training step, their stochastic-depth factors read as kernels would."""

    def __init__(self, rows):
        self.rows, self.read = rows, []

    def ptv3_train_bytes(self, net, levels, acts, fwd, bwd):
        for at in (acts, fwd, bwd):
            ctypes.c_size_t.from_address(at).value = 512
        return 0

    def _masks(self, masks):
        self.read.append([None if not at else list((ctypes.c_float * self.rows).from_address(at)) for at in masks])
        return 0

    def ptv3_train_fwd(self, net, levels, feat, dt, masks, *rest):
        return self._masks(masks)

    def ptv3_train_bwd(self, net, levels, dout, dt, masks, *rest):
        ctypes.memset(rest[3], 0, 4)   # the one gradient
        return self._masks(masks)


@pytest.fixture
def train_step(monkeypatch):
    """step(masks) -> rows of a step whose engine holds one parameter, over stand-ins for the library's two calls."""
    lib = _TrainLib(6)
    monkeypatch.setattr(native_train._lib, "load", lambda: lib)
    monkeypatch.setattr(native_train.ops, "_stream", lambda: None)
    weight = torch.nn.Parameter(torch.ones(1))
    engine = types.SimpleNamespace(net=native_train._Net(), out_channels=4, dtype=torch.float32,
                                   total=1, params=[weight], read_back=[weight])
    engine.versions = types.MethodType(native_train.TrainEngine.versions, engine)
    index = types.SimpleNamespace(levels=None)

    def step(masks):
        return native_train._Step.apply(engine, torch.zeros(6, 6), index, masks, weight)

    return types.SimpleNamespace(step=step, lib=lib, weight=weight, engine=engine)


@pytest.mark.parametrize("hooks", ["none", "copies", "misaligned copies"])
def test_backward_of_a_step_reads_the_masks_that_autograd_kept(hooks, train_step):
    """Saved-tensor hooks (checkpointing, offloading to the host) keep copies and let the originals go."""
    masks = [None, torch.arange(6.0).view(6, 1), None, torch.arange(6.0).neg().view(6, 1)]
    want = [None if m is None else m.flatten().tolist() for m in masks]

    def unpack(t):
        if hooks != "misaligned copies" or t.dim() < 2:
            return t
        return torch.cat([t.new_zeros(1, 1), t])[1:]

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), unpack) if hooks != "none" else contextlib.nullcontext():
        out = train_step.step(masks)
    if hooks != "none":
        for m in masks:     # what their memory holds once it has been handed out again
            if m is not None:
                m.fill_(7.0)
    del masks
    out.sum().backward()
    assert train_step.lib.read == [want, want]
    assert float(train_step.weight.grad) == 0.0


@pytest.mark.parametrize("change", [lambda t: t[:-1], lambda t: t.double(), lambda t: t.to("meta")], ids=["shorter", "dtype", "device"])
@pytest.mark.parametrize("which", [torch.uint8, torch.float32], ids=["activations", "masks"])
def test_backward_of_a_step_refuses_tensors_that_hooks_changed(change, which, train_step):
    """What the kernels would read past the end of, or where they cannot reach, is an error."""
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: change(t) if t.dtype == which else t):
        out = train_step.step([torch.ones(6, 1)])
    with pytest.raises(RuntimeError, match="saved-tensor hook"):
        out.sum().backward()
    assert len(train_step.lib.read) == 1      # the forward only


def test_backward_of_a_step_refuses_weights_written_since_its_forward(train_step):
    """The engine's copies of the weights follow the weights: the gradients would be those of another function."""
    out = train_step.step([None])
    with torch.no_grad():
        train_step.weight.mul_(2.0)
    again = train_step.step([None])
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    again.sum().backward()           # a step whose weights stand is not held up


def test_checkpointed_step_is_held_against_the_weights_it_was_computed_again_with(train_step):
    from torch.utils.checkpoint import checkpoint
    out = checkpoint(lambda: train_step.step([None]), use_reentrant=False)
    with torch.no_grad():
        train_step.weight.mul_(2.0)
    out.sum().backward()             # the forward ran again, with the weights as they are now
    assert len(train_step.lib.read) == 3


def _described(model):
    """A TrainEngine's description of a model on the CPU (nothing is launched; placement is not looked at)."""
    engine = native_train.TrainEngine.__new__(native_train.TrainEngine)
    engine.dtype, engine.device, engine.structure = torch.float16, torch.device("cpu"), native.Structure(model)
    engine._keep, engine._casts, engine._packs, engine._zero, engine.read_back = [], [], [], [], []
    engine.params, engine._placed, engine.total, engine._norms = [], set(), 0, []
    engine._describe(model, native.Parts(model))
    return engine


SMALL = dict(enc_depths=(1, 2, 1), enc_channels=(32, 64, 128), enc_num_head=(2, 4, 8), enc_patch_size=(64,) * 3, stride=(2, 2),
             dec_depths=(1, 1), dec_channels=(64, 64), dec_num_head=(4, 4), dec_patch_size=(64,) * 2)


def test_step_node_holds_the_parameters_it_writes_gradients_for_and_no_others():
    """A segmentation head or a mask token of a subclass is no part of the backbone's node: its gradient is not this node's
    to give."""
    from pointtransformerv3_amd import PointTransformerV3

    class Segmentor(PointTransformerV3):
        def __init__(self, **kw):
            super().__init__(**kw)
            self.mask_token = torch.nn.Parameter(torch.zeros(1, 6))
            self.head = torch.nn.Linear(64, 13)

    model = Segmentor(**SMALL)
    engine = _described(model)
    backbone = [p for part in (model.embedding, model.enc, model.dec) for p in part.parameters()]
    assert {id(p) for p in engine.params} == {id(p) for p in backbone} and len(engine.params) == len(backbone)
    assert engine.total == sum(p.numel() for p in backbone)


@pytest.mark.parametrize("share", ["block", "norm", "weight"])
def test_parameters_used_twice_are_left_to_the_modules(share):
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(**SMALL)
    a, b = model.enc.enc1.block0, model.enc.enc1.block1
    if share == "block":
        model.enc.enc1.block1 = a
    elif share == "norm":
        b.norm2 = a.norm1
    else:
        b.mlp[0].fc1.weight = a.mlp[0].fc1.weight
    with pytest.raises(native.Unsupported):
        _described(model)


def _set(path, value):
    """A change of one attribute: path is its owner within enc.enc1 and its name."""
    def change(stage):
        *owner, name = path.split(".")
        at = stage
        for key in owner:
            at = at[int(key)] if key.isdigit() else getattr(at, key)
        setattr(at, name, value(getattr(at, name)) if callable(value) and not isinstance(value, torch.nn.Module) else value)
    return change


def _replace_forward(stage):
    stage.block0.mlp[0].forward = lambda x: x


def _transposed(stage):
    w = stage.block0.attn.proj.weight
    w.data = w.data.t()                   # the same address, another matrix


def _narrowed(stage):
    w = stage.block0.mlp[0].fc1.weight
    w.data = w.data[:16]


def _same_data(stage):
    lin = stage.block0.mlp[0].fc2
    lin.weight = torch.nn.Parameter(lin.weight.data)


CHANGES = dict(
    norm_eps=_set("block0.norm1.0.eps", 1e-3), batch_norm_eps=_set("down.norm.0.eps", 0.1), scale=_set("block0.attn.scale", 0.5),
    patch_size=_set("block0.attn.patch_size", 32), order_index=_set("block1.attn.order_index", 2), heads=_set("block0.attn.num_heads", 8),
    flash=_set("block0.attn.enable_flash", False), attn_drop=_set("block0.attn.attn_drop", 0.1),
    proj_drop=_set("block0.attn.proj_drop.p", 0.1), mlp_drop=_set("block1.mlp.0.drop.p", 0.1),
    gelu=_set("block0.mlp.0.act.approximate", "tanh"), pre_norm=_set("block0.pre_norm", False),
    shuffle_orders=_set("down.shuffle_orders", False), reduce=_set("down.reduce", "mean"), traceable=_set("down.traceable", False),
    plan_kernel_sizes=_set("down.plan_kernel_sizes", (5,)), track=_set("down.norm.0.track_running_stats", False),
    forward=_replace_forward, child_added=lambda st: st.add(torch.nn.ReLU(), name="extra"),
    child_removed=lambda st: st._modules.pop("block1"), child_replaced=lambda st: st.block0.drop_path._modules.update({"0": torch.nn.Dropout(0.5)}),
    bias_gone=_set("block0.mlp.0.fc1.bias", None), norm_without_weight=_set("block0.norm2.0.weight", None),
    statistics_gone=_set("down.norm.0.running_var", None), counter_replaced=_set("down.norm.0.num_batches_tracked", lambda t: t.clone()),
    statistics_replaced=_set("down.norm.0.running_mean", lambda t: t.clone()), parameter_replaced=_same_data,
    data_replaced=lambda st: setattr(st.block0.attn.qkv.weight, "data", st.block0.attn.qkv.weight.data.clone()),
    data_transposed=_transposed, data_narrowed=_narrowed,
    attribute_gone=lambda st: delattr(st.block0.attn, "scale"), scale_no_number=_set("block0.attn.scale", torch.tensor(0.5)),
)


@pytest.mark.parametrize("name", sorted(CHANGES))
def test_structure_notices_what_the_modules_would_act_on(name):
    """What was read when the model was described is compared at every forward; nothing of it raises."""
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(**SMALL)
    structure = native.Structure(model)
    assert structure.why is None and structure.same() and structure.same()
    CHANGES[name](model.enc.enc1)
    assert structure.same() is False
    again = native.Structure(model)
    assert again.same()
    if name in ("forward", "attribute_gone", "scale_no_number"):
        assert again.why is not None      # left to the modules whatever they make of it


def test_number_of_orders_belongs_to_the_structure_but_their_names_do_not():
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(order=["z", "hilbert"], **SMALL)
    structure = native.Structure(model)
    model.order = ["hilbert", "z-trans"]
    assert structure.same()
    model.order.append("z")
    assert not structure.same()


def test_step_follows_a_momentum_schedule():
    """A BatchNorm's momentum is read at every step; a cumulative average (None) is left to the modules."""
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(**SMALL)
    engine = _described(model)
    norms = [m for m in model.modules() if isinstance(m, torch.nn.BatchNorm1d)]
    assert sorted(map(id, norms)) == sorted(id(m) for _, m in engine._norms)
    places = [engine.net.stem.bn] + [engine.net.stage[s].pool_bn for s in (1, 2)]
    places += [b for s in (0, 1) for b in (engine.net.stage[s].up_bn, engine.net.stage[s].up_skip_bn)]
    for i, m in enumerate(norms):
        m.momentum = 0.1 + 0.05 * i
    assert engine.averaging()
    engine.follow_momentum()
    got = sorted(round(d.momentum, 4) for d in places)
    assert got == [round(0.1 + 0.05 * i, 4) for i in range(len(norms))]
    norms[1].momentum = None
    assert not engine.averaging()


def test_a_described_or_refused_model_is_let_go():
    """The tables of engines are keyed by the model: what they hold must not hold it."""
    from pointtransformerv3_amd import PointTransformerV3
    for table, make in ((native._ENGINES, lambda m: native.Refused(m, "for the test")),
                        (native_train._ENGINES, lambda m: native.Refused(m, "for the test")), (native_train._ENGINES, _engine_of)):
        model = PointTransformerV3(**SMALL)
        table.setdefault(model, {})["held"] = make(model)
        seen, weight = weakref.ref(model), weakref.ref(model.enc.enc1.block0.attn.qkv.weight)
        before = len(table)
        del model
        gc.collect()
        assert seen() is None and weight() is None and len(table) == before - 1


def _engine_of(model):
    return _described(model)


class _OwnStem(torch.nn.Module):
    def forward(self, point):
        return point


def _without(*names):
    def change(model):
        for name in names:
            at, key = (model.get_submodule(name.rpartition(".")[0]), name.rpartition(".")[2])
            delattr(at, key)
    return change


FOREIGN = dict(
    own_embedding=lambda m: setattr(m, "embedding", _OwnStem()), no_embedding=_without("embedding"), no_encoder=_without("enc"),
    no_decoder=_without("dec"), no_stem_norm=_without("embedding.stem.norm"), no_mlp=_without("enc.enc1.block0.mlp"),
    no_attention=_without("dec.dec0.block0.attn"), no_projection=_without("enc.enc1.block0.attn.proj"),
    own_norm=lambda m: setattr(m.enc.enc1.down, "norm", torch.nn.LayerNorm(64)), no_norm=lambda m: setattr(m.enc.enc1.down, "norm", None),
    no_pool_projection=_without("enc.enc1.down.proj"), identity=lambda m: setattr(m.dec.dec0.up, "proj", torch.nn.Identity()),
    nothing=lambda m: [_without(n)(m) for n in ("embedding", "enc", "dec")], row=_set("enc.enc1.block0.attn.order_index", 7),
    reduce=_set("enc.enc1.down.reduce", "median"), strides=_set("stride", (2,)),
    pruned=lambda m: setattr(m.enc.enc1.block0.mlp[0].fc1.weight, "data", m.enc.enc1.block0.mlp[0].fc1.weight.data[:64]),
    pruned_norm=lambda m: setattr(m.enc.enc1.block0.norm1[0].weight, "data", torch.ones(32)),
    heads=_set("enc.enc1.block0.attn.num_heads", 0), order_set=_set("order", {"z"}), order_gone=_without("order"),
    order_iterator=lambda m: setattr(m, "order", iter(["z", "hilbert"])),
)


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("name", sorted(FOREIGN))
def test_models_of_another_architecture_are_left_to_the_modules(name, train, monkeypatch):
    """What the native paths do not cover is the modules' to run or to refuse: looking at it raises nothing."""
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(**SMALL).train(train)
    FOREIGN[name](model)
    with pytest.raises(native.Unsupported):
        native.Parts(model)
        _described(model)
    monkeypatch.setattr(native, "plain_inputs", lambda data: True)
    data = dict(feat=torch.zeros(4, 6), grid_coord=torch.zeros(4, 3, dtype=torch.int32), offset=torch.tensor([4]))
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *a: train)
    with torch.set_grad_enabled(train):
        for _ in range(2):
            assert (native_train if train else native).engine_for(model, data) is None


@pytest.mark.parametrize("n", [1, 2000, 400_000])
def test_index_tables_are_apart_from_the_scratch(n):
    """The buffer that a returned Point's sparse indices lie in holds little else; voxel hash, keys and counts are another."""
    from pointtransformerv3_amd import _lib, levels
    cfg = levels.Cfg(n=n, n_levels=5, n_orders=4, n_scenes=4, stem5=1, patch=(ctypes.c_int32 * 8)(*[1024] * 8))
    tables, scratch = ctypes.c_size_t(), ctypes.c_size_t()
    lib = _lib.load()
    assert lib.ptv3_index_begin_bytes(ctypes.byref(cfg), ctypes.byref(tables), ctypes.byref(scratch)) == 0
    assert 16 * n <= tables.value <= 16 * n + 4096 and scratch.value >= 100 * n
    assert lib.ptv3_index_begin_bytes(ctypes.byref(cfg), None, ctypes.byref(scratch)) != 0


def test_rule_of_convolutions_that_no_tile_form_takes():
    """Few pairs and small dense volumes: float rows; larger dense volumes: the neighbour map; else half rows. Float: pair
    rows unless a dense volume's would take more than 32 GiB."""
    from pointtransformerv3_amd import _lib, ops
    form = _lib.load().ptv3_conv_pair_form
    f32, f16 = ops.DTYPE_CODES[torch.float32], ops.DTYPE_CODES[torch.float16]
    few = _lib.load().ptv3_conv_few_pairs
    for c in (64, 128):
        line = max(p for p in range(1000, 400_000, 1000) if few(p, c))
        assert form(f16, 10_000_000, line, 27, c, c, 0.6) == form(f16, line // 27, line, 27, c, c, 0.6) == ops.CONV_PAIRS_WIDE
        assert form(f16, 10_000_000, line + 1000, 27, c, c, 0.6) == ops.CONV_PAIRS
    for c in (32, 256, 512):
        assert form(f16, 1000, 16_000, 27, c, c, 0.6) == ops.CONV_PAIRS
        assert form(f16, 1000, 16_300, 27, c, c, 0.6) == form(f16, 9000, 229_500, 27, c, c, 0.6) == ops.CONV_PAIRS_WIDE
        assert form(f16, 9000, 229_501, 27, c, c, 0.6) == ops.CONV_DENSE
        assert form(f16, 9000, 229_501, 27, c, c, 1.0) == ops.CONV_PAIRS
    assert form(f16, 9000, 1_000_000, 125, 16, 32, 0.6) == ops.CONV_PAIRS_WIDE
    assert form(f16, 12_000, 1_100_000, 125, 16, 32, 0.6) == ops.CONV_DENSE
    assert form(f16, 1000, 20_000, 27, 48, 96, 0.6) == ops.CONV_DENSE      # no float rows of this shape
    assert form(f16, 1000, 2_000, 27, 32, 12, 0.6) == ops.CONV_DENSE       # outputs not in 8s
    assert form(f32, 10_000_000, 27 * 10_000_000, 27, 31, 31, 0.6) == ops.CONV_PAIRS
    assert form(f32, 10_000_000, 27 * 10_000_000, 27, 32, 32, 0.6) == ops.CONV_DENSE
    assert form(f32, 100_000_000, 27 * 10_000_000, 27, 512, 512, 0.6) == ops.CONV_PAIRS
    assert form(f16, 0, 0, 27, 32, 32, 0.6) == ops.CONV_PAIRS


@pytest.mark.parametrize("when", ["before", "after"])
@pytest.mark.parametrize("kind", [native.SerializedAttention, native.Block, torch.nn.Linear])
def test_a_class_whose_forward_was_replaced_is_left_to_the_modules(kind, when, monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3
    model = PointTransformerV3(**SMALL)
    structure = native.Structure(model)
    monkeypatch.setattr(kind, "forward", lambda self, x: x)
    if when == "after":
        assert not structure.same()
    else:
        assert native.Structure(model).why is not None
    monkeypatch.undo()
    assert structure.same() and native.Structure(model).why is None


def _attention_cut(items, slots, n_seq, max_seqlen=1024, cus=256):
    from pointtransformerv3_amd import _lib
    full = ctypes.c_int64(-1)
    split = _lib.load().ptv3_patch_attn_cut(items, slots, n_seq, max_seqlen, cus, ctypes.byref(full))
    return full.value, split


@pytest.mark.parametrize("cus", [256, 80, 6])
@pytest.mark.parametrize("mean", [1, 131, 600, 1024])
def test_attention_cut_fills_every_xcd_alike(mean, cus):
    """Ranges that are meant to have a CU each do: counted where the kernel puts them, an eighth of the items on an XCD."""
    for items in [*range(1, 1400), 4000, 100_000]:
        full, split = _attention_cut(items, mean * items, items, cus=cus)
        assert 1 <= split <= 8 and (full == items if split == 1 else full == (0 if items <= cus else items // cus * cus))
        if split > 1:
            fullest = -(-(-(-(items - full) // 8) * split) // max(cus // 8, 1))
            assert fullest <= split     # never more on a CU than an item
            assert fullest == 1 or -(-mean // 32) >= 7 * split


@pytest.mark.parametrize("items,mean,want", [(42, 981, (0, 5)), (84, 976, (0, 2)), (340, 1024, (256, 2)), (554, 1024, (512, 5)),
                                             (1108, 1024, (1024, 2)), (192, 250, (192, 1)), (416, 238, (416, 1)), (256, 723, (0, 2)),
                                             (256, 804, (0, 2)), (256, 486, (256, 1)), (256, 1024, (256, 1)), (198, 1024, (0, 2)),
                                             (232, 1024, (0, 2)), (312, 1024, (256, 4)), (4, 1024, (0, 8)), (512, 723, (512, 1))])
def test_attention_cut_measured(items, mean, want):
    assert _attention_cut(items, mean * items, items) == want


def test_rules_that_fill_the_part_ask_the_device_for_its_cus(tmp_path):
    """On a quarter of the part (64 CUs, as one that is divided shows them) a rule decides as on the whole one for four times
    the voxels. The device is a library that answers in the runtime's place; on the host the library's own answer is 256."""
    import os
    import shutil
    import subprocess
    import sys

    from pointtransformerv3_amd import _lib
    if shutil.which("gcc") is None:
        pytest.skip("no C compiler")
    src, so = tmp_path / "quarter.c", tmp_path / "quarter.so"
    src.write_text("int hipGetDevice(int *d) { *d = 0; return 0; }\n"
                   "int hipDeviceGetAttribute(int *v, int what, int dev) { *v = 64; return 0; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    voxels = list(range(384, 60_000, 384))
    code = ("import ctypes, sys\n"
            f"ctypes.CDLL({str(so)!r}, mode=ctypes.RTLD_GLOBAL)\n"
            f"lib, i64 = ctypes.CDLL({_lib.LIB_PATH!r}), ctypes.c_int64\n"
            f"v = {voxels}\n"
            "print([lib.ptv3_conv_tile_voxels(i64(n), 128) for n in v], [lib.ptv3_conv_form(i64(n), i64(9 * n + 70_000), 64) for n in v])")
    out = subprocess.run([sys.executable, "-c", code], check=True, capture_output=True, text=True, env=dict(os.environ)).stdout
    lib = _lib.load()
    tiles, form = [lib.ptv3_conv_tile_voxels(4 * n, 128) for n in voxels], [lib.ptv3_conv_form(4 * n, 4 * (9 * n + 70_000), 64) for n in voxels]
    if not torch.cuda.is_available() or torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert {96, 128} == set(tiles) and {1, 2} == set(form)
        assert out.split("\n")[0] == f"{tiles} {form}"
