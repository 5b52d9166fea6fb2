"""A training step's forward and backward from native code (ptv3_train_fwd / ptv3_train_bwd): under half-precision
autocast the whole feature side of a PointTransformerV3 is one autograd node. Module by module the same step is some 250
Python autograd functions each way and about 20 ms of host time whatever the batch. Takes the default architecture in
training mode (see native.Parts, TrainEngine); anything else goes through the modules (model.py), which stay the
definition of the result.

The parameter gradients are views of one flat buffer and all come at the end of the backward: a reducer that wants to
overlap them with it has nothing to start on before (a hook on any submodule, which sends the step through the modules,
gives them one by one), and a p.grad that is kept or saved keeps the buffer, 185 MB for the default model (its clone does
not)."""
import ctypes
import weakref

import torch
import torch.nn as nn

from . import _lib, levels, native, ops
from .modules import DropPath
from .native import Parts, Structure, Unsupported, _need
from .point import AttrDict, Point, batch2offset

_i32, _i64, _f32, _ptr = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p


class _Linear(ctypes.Structure):
    _fields_ = [("w", _ptr), ("wt", _ptr), ("b", _ptr), ("cin", _i32), ("cout", _i32), ("gw", _i64), ("gb", _i64)]


class _Norm(ctypes.Structure):
    _fields_ = [("g", _ptr), ("b", _ptr), ("eps", _f32), ("reserved", _i32), ("gg", _i64), ("gb", _i64)]


class _Bn(ctypes.Structure):
    _fields_ = [("g", _ptr), ("b", _ptr), ("g16", _ptr), ("b16", _ptr), ("running_mean", _ptr), ("running_var", _ptr),
                ("eps", _f32), ("momentum", _f32), ("gg", _i64)]


class _Block(ctypes.Structure):
    _fields_ = [("channels", _i32), ("heads", _i32), ("row", _i32), ("reserved", _i32), ("scale", _f32), ("reserved2", _f32),
                ("conv_w", _ptr), ("conv_b", _ptr), ("conv_mirror", _ptr), ("conv_packed", _ptr), ("conv_mirror_packed", _ptr),
                ("g_conv_w", _i64), ("g_conv_b", _i64),
                ("cpe", _Linear), ("qkv", _Linear), ("proj", _Linear), ("fc1", _Linear), ("fc2", _Linear),
                ("ln_cpe", _Norm), ("ln1", _Norm), ("ln2", _Norm)]


class _Stage(ctypes.Structure):
    _fields_ = [("channels", _i32), ("dec_channels", _i32), ("n_enc", _i32), ("n_dec", _i32), ("pool_reduce", _i32),
                ("reserved", _i32), ("enc", _ptr), ("dec", _ptr), ("pool", _Linear), ("up", _Linear), ("up_skip", _Linear),
                ("pool_bn", _Bn), ("up_bn", _Bn), ("up_skip_bn", _Bn)]


class _Stem(ctypes.Structure):
    _fields_ = [("w", _ptr), ("cin", _i32), ("cin_padded", _i32), ("gw", _i64), ("bn", _Bn)]


class _Net(ctypes.Structure):
    _fields_ = [("dtype", _i32), ("n_stages", _i32), ("patch", _i32 * levels.MAX_LEVELS),
                ("max_pair_density", _f32), ("reserved2", _f32), ("stem", _Stem), ("zero", _ptr),
                ("n_zero", _i32), ("has_side", _i32), ("zero_blocks", _i64), ("stage", _Stage * levels.MAX_LEVELS), ("side", _ptr)]


class TrainEngine(native.Copies):
    """Describes one model (float masters) for training under autocast to `dtype`."""

    def __init__(self, model, dtype):
        super().__init__()
        self.structure = Structure(model)
        _need(self.structure.why is None, self.structure.why)
        parts = Parts(model)
        self.dtype = dtype
        self.device = self.structure.tensors[0].device
        _need(all(p.is_cuda and p.device == self.device and p.is_contiguous() and p.dtype == torch.float32
                  for p in self.structure.tensors), "float weights on one GPU")
        _need(not model.cls_mode, "the encoder-only model hands out intermediate features")
        _need(not any(p.is_inference() for p in self.structure.tensors), "inference tensors")
        self._casts, self._packs, self._zero = [], [], []
        self.read_back = []             # parameters whose values the backward reads, itself or as a copy made by the forward
        # the parameters of the step's node, in the order their gradients lie in the flat buffer: those that the
        # description places, each of which the backward writes once and in whole. A subclass may hold more (a head, a
        # mask token): they are no part of this node
        self.params, self._placed, self.total = [], set(), 0
        self._norms = []                # (its ptv3 description, module): the momentum may follow a schedule
        self._describe(model, parts)
        self._finish()
        # the weight gradients' stream; whatever is queued on it the backward's own stream waits for before the call returns
        self.side = torch.cuda.Stream(self.device)
        self.net.has_side, self.net.side = 1, self.side.cuda_stream
        self.batches = [m.num_batches_tracked for m in self.structure.modules
                        if isinstance(m, nn.BatchNorm1d) and m.num_batches_tracked is not None]

    def _buffer(self, elements):
        t = torch.empty(elements, dtype=self.dtype, device=self.device)
        self._keep.append(t)
        return t.data_ptr()

    def _copy(self, t, layout="plain"):
        """Address of the parameter's copy in the compute dtype (ops.cast_cached's layouts)."""
        shape, _ = ops._cast_shape(t, layout)
        dst = self._buffer(t.numel())
        self._casts.append((t, dst, shape, int(layout != "plain")))
        return dst

    def _at(self, p):
        """Place of the parameter's gradient. Gradients are written, not added up: a parameter has one place."""
        _need(p not in self._placed, "a parameter that is used twice")
        self._placed.add(p)
        self.params.append(p)
        at = self.total
        self.total += p.numel()
        return at

    def versions(self):
        return [p._version for p in self.read_back]

    def _linear(self, m, cin, cout):
        native.check_linear(m, cin, cout)
        self.read_back.append(m.weight)
        return _Linear(self._copy(m.weight), self._copy(m.weight, "transpose"), self._copy(m.bias), cin, cout,
                       self._at(m.weight), self._at(m.bias))

    def _norm(self, m, c):
        native.check_layer_norm(m, c)
        gg, gb = self._at(m.weight), self._at(m.bias)
        self._zero += [(gg, c), (gb, c)]
        self.read_back.append(m.weight)
        return _Norm(m.weight.data_ptr(), m.bias.data_ptr(), m.eps, 0, gg, gb)

    def _bn(self, m, c):
        native.check_batch_norm(m, c)
        gg, gb = self._at(m.weight), self._at(m.bias)   # the kernel writes both, one behind the other
        assert gb == gg + c
        self.read_back += [m.weight, m.bias]
        return _Bn(m.weight.data_ptr(), m.bias.data_ptr(), self._copy(m.weight), self._copy(m.bias), m.running_mean.data_ptr(),
                   m.running_var.data_ptr(), m.eps, 0.0, gg)

    def _block(self, b, c):
        conv, attn, mlp = b.cpe[0], b.attn, b.mlp[0]
        _need(attn.attn_drop == 0 and attn.proj_drop.p == 0 and mlp.drop.p == 0 and c // attn.num_heads == 16, "dropout or head size")
        d = _Block(channels=c, heads=attn.num_heads, row=attn.order_index, scale=attn.scale)
        self.read_back.append(conv.weight)
        d.conv_w, d.conv_b, d.conv_mirror = self._copy(conv.weight), self._copy(conv.bias), self._copy(conv.weight, "mirror")
        if c in native.CONV_PACKED:
            d.conv_packed, d.conv_mirror_packed = self._buffer(27 * c * c), self._buffer(27 * c * c)
            self._packs += [(d.conv_w, d.conv_packed, c, 27), (d.conv_mirror, d.conv_mirror_packed, c, 27)]
        d.g_conv_w, d.g_conv_b = self._at(conv.weight), self._at(conv.bias)
        d.cpe, d.qkv, d.proj = self._linear(b.cpe[1], c, c), self._linear(attn.qkv, c, 3 * c), self._linear(attn.proj, c, c)
        d.fc1, d.fc2 = self._linear(mlp.fc1, c, 4 * c), self._linear(mlp.fc2, 4 * c, c)
        d.ln_cpe, d.ln1, d.ln2 = self._norm(b.cpe[2], c), self._norm(b.norm1[0], c), self._norm(b.norm2[0], c)
        return d

    def _describe(self, model, p):
        _need(all(st.enc for st in p.stages) and all(st.dec for st in p.stages[:-1]), "a stage without blocks")
        net = self.net = _Net(dtype=ops.DTYPE_CODES[self.dtype], n_stages=len(p.stages), max_pair_density=self.structure.density)
        conv = p.stem_conv
        padded = -(-conv.in_channels // 16) * 16
        net.stem.w = self._buffer(conv.out_channels * 125 * padded)
        net.stem.cin, net.stem.cin_padded, net.stem.gw = conv.in_channels, padded, self._at(conv.weight)
        net.stem.bn = self._bn(p.stem_bn, conv.out_channels)
        self._norms.append((net.stem.bn, p.stem_bn))
        self._refresh = native._Refresh(dtype=net.dtype, stem_src=self._copy(conv.weight), stem_dst=net.stem.w,
                                        stem_rows=conv.out_channels * 125, stem_in=conv.in_channels, stem_padded=padded)
        self.drops, below = [], conv.out_channels
        for s, st in enumerate(p.stages):
            d = net.stage[s]
            d.channels, d.n_enc, d.dec_channels, d.n_dec = st.channels, len(st.enc), st.dec_channels, len(st.dec)
            if st.down is not None:
                d.pool, d.pool_bn = self._linear(st.down.proj, below, st.channels), self._bn(st.bn, st.channels)
                d.pool_reduce = ops.REDUCE_OPS[st.down.reduce]
                self._norms.append((d.pool_bn, st.bn))
            if st.up is not None:
                d.up = self._linear(st.up.proj[0], st.up.proj[0].in_features, st.dec_channels)
                d.up_skip = self._linear(st.up.proj_skip[0], st.channels, st.dec_channels)
                d.up_bn, d.up_skip_bn = self._bn(st.up.proj[1], st.dec_channels), self._bn(st.up.proj_skip[1], st.dec_channels)
                self._norms += [(d.up_bn, st.up.proj[1]), (d.up_skip_bn, st.up.proj_skip[1])]
            for attr, bs, c in (("enc", st.enc, st.channels), ("dec", st.dec, st.dec_channels)):
                if bs:
                    arr = (_Block * len(bs))(*[self._block(b, c) for b in bs])
                    self._keep.append(arr)
                    setattr(d, attr, ctypes.addressof(arr))
            net.patch[s] = st.patch
            below = st.channels
        order = [(s, b) for s, st in enumerate(p.stages) for b in st.enc]
        order += [(s, b) for s in reversed(range(len(p.stages) - 1)) for b in p.stages[s].dec]
        self.drops = [(s, b.drop_path[0]) for s, b in order]
        self.out_channels = p.stages[0].dec_channels
        self.layout = p.layout(model)
        form, widths = _lib.load().ptv3_conv_form, p.widths()

        def want(level, v):
            flags = levels.PAIRS5 | levels.PAIR_OUT5 if level == 0 else 0
            for c in widths[level]:
                flags |= levels.TILES if form(v.n, v.n_pairs, c) else levels.PAIRS
                flags |= levels.PAIRS | levels.PAIR_OUT
            return flags

        self.want = want

    def _finish(self):
        lib, r = _lib.load(), self._refresh
        rows, at = [], 0
        for t, dst, (a, b, c), mirror in self._casts:
            rows.append((t.data_ptr(), dst, a, b, c, mirror, at))
            at += lib.ptv3_cast_params_blocks(a, b, c, mirror)
        r.cast, r.n_cast, r.cast_blocks = self._table(rows, ops._CAST_JOB), len(rows), at
        rows, at = [], 0
        for src, dst, c, taps in self._packs:
            rows.append((src, dst, c, taps, at))
            at += lib.ptv3_subm_conv_pack_weight_blocks(c, taps)
        r.conv, r.n_conv, r.conv_blocks = self._table(rows, ops._PACK_JOB), len(rows), at
        rows, at = [], 0
        for start, count in self._zero:
            rows.append((start, count, at))
            at += -(-count // 256)
        net = self.net
        net.zero, net.n_zero, net.zero_blocks = self._table(rows, [("at", "<i8"), ("count", "<i8"), ("block", "<i8")]), len(rows), at

    def _table(self, rows, dtype):
        t = native.job_table(rows, dtype, self.device)
        self._keep.append(t)
        return t.data_ptr() if t is not None else None

    def averaging(self):
        """Whether the running statistics follow an exponential average (momentum None: a cumulative one)."""
        return all(m.momentum is not None for _, m in self._norms)

    def follow_momentum(self):
        for d, m in self._norms:
            d.momentum = m.momentum

    def masks(self, sizes):
        """The stochastic-depth row factors in the order the blocks would draw them (DropPath.mask; model.py:602-604)."""
        out, keeps, drawn = [], [], []
        for s, drop in self.drops:
            rate = drop.drop_prob if isinstance(drop, DropPath) else 0.0
            for _ in range(2):
                if rate == 0.0:
                    out.append(None)
                    continue
                m = torch.empty((sizes[s].n, 1), dtype=self.dtype, device=self.device).bernoulli_(1.0 - rate)
                if drop.scale_by_keep and rate < 1.0:
                    drawn.append(m)
                    keeps.append(1.0 - rate)
                out.append(m)
        if drawn:
            torch._foreach_div_(drawn, keeps)
        return out

    def forward(self, model, data):
        feat = data["feat"].detach().contiguous()
        point = Point.__new__(Point)
        dict.update(point, data)
        grid, offset, batch = native.coordinates(point)

        masks = []

        def sized(sizes):
            if any(v.n < 2 for v in sizes):
                return
            # float masters are cast, transposed and packed once per step: here, where the host draws the masks with some
            # 45 small launches and the GPU would wait for them (2 x 15k voxels 7.79 -> 7.72 ms against in front of the sort)
            _lib.check(_lib.load().ptv3_net_refresh(ctypes.byref(self._refresh), ops._stream()), "ptv3_net_refresh")
            if self.batches:
                torch._foreach_add_(self.batches, 1)
            masks.extend(self.masks(sizes))

        self.follow_momentum()
        self.used_here()
        model._prologue_state = None
        index = levels.build(self.layout, grid, offset, batch, list(model.order), model.shuffle_orders, self.want, sized=sized)
        if any(v.n < 2 for v in index.levels):
            raise ValueError("Expected more than 1 value per channel when training")   # as BatchNorm1d does
        out = _Step.apply(self, feat, index, masks, *self.params)
        point["batch"] = index.batch
        native.fill_point(point, index, 0, out, self.net.patch[0])
        return point


def _addresses(tensors):
    return (_ptr * len(tensors))(*[None if t is None else t.data_ptr() for t in tensors])


def _train_bytes(net, index_levels):
    """Bytes of the activations, the forward's scratch and the backward's."""
    sizes = (ctypes.c_size_t * 3)()
    at = ctypes.addressof(sizes)
    _lib.check(_lib.load().ptv3_train_bytes(ctypes.byref(net), index_levels, at, at + 8, at + 16), "ptv3_train_bytes")
    return list(sizes)


class _Step(torch.autograd.Function):
    @staticmethod
    def forward(ctx, engine, feat, index, masks, *params):
        lib = _lib.load()
        u8 = dict(dtype=torch.uint8, device=feat.device)
        sizes = _train_bytes(engine.net, index.levels)
        acts, scratch = torch.empty(sizes[0], **u8), torch.empty(sizes[1], **u8)
        out = torch.empty((feat.shape[0], engine.out_channels), dtype=torch.float32, device=feat.device)
        _lib.check(lib.ptv3_train_fwd(ctypes.byref(engine.net), index.levels, feat.data_ptr(), ops.DTYPE_CODES[feat.dtype],
                                      _addresses(masks), acts.data_ptr(), scratch.data_ptr(), sizes[1], out.data_ptr(), ops._stream()), "ptv3_train_fwd")
        ctx.engine, ctx.index, ctx.scratch_bytes = engine, index, sizes[2]
        ctx.acts_bytes, ctx.masked = sizes[0], [0 if m is None else m.numel() for m in masks]
        # freed by autograd after the backward, as the activations of separate nodes would be; the versions go with them, so
        # that activations which a checkpoint computes again are held against the weights they were computed with
        ctx.save_for_backward(acts, torch.tensor(engine.versions()), *[m for m in masks if m is not None])
        return out

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dout):
        engine, index = ctx.engine, ctx.index
        # under saved-tensor hooks (checkpointing, offloading) these are not the tensors of the forward but what the hooks
        # made of them: every address is taken here, and the views the kernels assume are made sure of
        acts, versions, *kept = ctx.saved_tensors
        # the weights' copies are the engine's and follow the weights at every forward, so a weight that was written since
        # this step's forward is an error, as it is where every node saves its own
        if versions.tolist() != engine.versions():
            raise RuntimeError("one of the variables needed for gradient computation has been modified by an inplace operation: "
                               "a parameter of PointTransformerV3 was written between a training step's forward and its backward")
        want = [(torch.uint8, ctx.acts_bytes)] + [(engine.dtype, n) for n in ctx.masked if n]
        for t, (dtype, numel) in zip((acts, *kept), want):
            if t.device != dout.device or t.dtype != dtype or t.numel() != numel:
                raise _lib.Ptv3Error("a saved-tensor hook handed back another tensor than it was given: "
                                     f"{t.numel()} x {t.dtype} on {t.device}, not {numel} x {dtype} on {dout.device}")
        acts, *kept = [t if t.is_contiguous() and t.data_ptr() % 256 == 0 else t.clone(memory_format=torch.contiguous_format)
                       for t in (acts, *kept)]
        kept = iter(kept)
        masks = [next(kept) if masked else None for masked in ctx.masked]
        dout = dout.contiguous()
        grads = torch.empty(engine.total, dtype=torch.float32, device=dout.device)
        net, nbytes = engine.net, ctx.scratch_bytes
        try:
            scratch = torch.empty(nbytes, dtype=torch.uint8, device=dout.device)
        except torch.cuda.OutOfMemoryError:
            # what the weight gradients read is held twice for the sake of the second stream: at 4 x 100k voxels 2.1 GiB of
            # scratch, 1.5 without
            net = type(net).from_buffer_copy(net)
            net.side = None
            nbytes = _train_bytes(net, index.levels)[2]
            scratch = torch.empty(nbytes, dtype=torch.uint8, device=dout.device)
        _lib.check(_lib.load().ptv3_train_bwd(ctypes.byref(net), index.levels, dout.data_ptr(), ops.DTYPE_CODES[dout.dtype],
                                              _addresses(masks), acts.data_ptr(), scratch.data_ptr(), nbytes,
                                              grads.data_ptr(), ops._stream()), "ptv3_train_bwd")
        views = torch._utils._unflatten_dense_tensors(grads, engine.params)
        needed = ctx.needs_input_grad[4:]
        return (None,) * 4 + tuple(g if need else None for g, need in zip(views, needed))


_ENGINES = weakref.WeakKeyDictionary()   # model -> {dtype: TrainEngine or native.Refused}, as native._ENGINES


def engine_for(model, data):
    """The TrainEngine that computes model(data), or None: the modules do."""
    if not (model.training and torch.is_grad_enabled() and torch.is_autocast_enabled()) or model.cls_mode:
        return None
    dtype = torch.get_autocast_dtype("cuda")
    if dtype not in (torch.float16, torch.bfloat16) or not native.plain_inputs(data) or data["feat"].requires_grad:
        return None
    held = _ENGINES.setdefault(model, {})
    engine = held.get(dtype)
    if engine is None or not engine.structure.same():
        try:
            engine = TrainEngine(model, dtype)
        except Unsupported as e:
            engine = native.Refused(model, str(e))
        held[dtype] = engine
    if isinstance(engine, native.Refused) or data["feat"].shape[1] != engine.net.stem.cin or data["feat"].shape[0] < 2:
        return None
    if data["feat"].device != engine.device:
        return None
    if engine.structure.hooked() or not all(m.training for m in engine.structure.flagged):
        return None
    return engine if engine.averaging() and any(p.requires_grad for p in engine.params) else None
