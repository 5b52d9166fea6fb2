"""The inference forward of a PointTransformerV3 from native code: the index by ptv3_index_* (levels.py), the features by one
ptv3_features_fwd call over a description of the model's weights (ptv3_net). Module by module the same launches cost the
host about 5 ms per forward; described once and queued natively they cost about a tenth of that.

An Engine describes one model in one compute dtype. It takes the default architecture (see Engine._describe); any other
model, a model with hooks or submodules in training mode, and inputs that carry tables of their own go through the
modules (model.py), which stay the definition of the result."""
import ctypes
import itertools
import operator
import weakref

import numpy as np
import torch
import torch.nn as nn

from . import _lib, levels, ops
from .modules import (MLP, Block, DropPath, Embedding, LayerNorm, PointSequential, SerializedAttention, SerializedPooling,
                      SerializedUnpooling)
from .point import AttrDict, Point, batch2offset
from .sparse import SparseConvTensor, SubMConv3d

_i32, _i64, _f32, _ptr = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p


class _Linear(ctypes.Structure):
    _fields_ = [("w", _ptr), ("b", _ptr), ("cin", _i32), ("cout", _i32)]


class _Norm(ctypes.Structure):
    _fields_ = [("g", _ptr), ("b", _ptr), ("eps", _f32), ("reserved", _i32)]


class _Bn(ctypes.Structure):
    _fields_ = [("mean", _ptr), ("var", _ptr), ("g", _ptr), ("b", _ptr), ("eps", _f32), ("stats_f32", _i32)]


class _Block(ctypes.Structure):
    _fields_ = [("channels", _i32), ("heads", _i32), ("row", _i32), ("reserved", _i32), ("scale", _f32), ("reserved2", _f32),
                ("conv_w", _ptr), ("conv_b", _ptr), ("conv_packed", _ptr),
                ("cpe", _Linear), ("qkv", _Linear), ("proj", _Linear), ("fc1", _Linear), ("fc2", _Linear),
                ("ln_cpe", _Norm), ("ln1", _Norm), ("ln2", _Norm),
                ("mlp_packed", _ptr), ("proj_packed", _ptr), ("head_packed", _ptr)]


class _Stage(ctypes.Structure):
    _fields_ = [("channels", _i32), ("dec_channels", _i32), ("n_enc", _i32), ("n_dec", _i32), ("pool_reduce", _i32),
                ("reserved", _i32), ("enc", _ptr), ("dec", _ptr), ("pool", _Linear), ("up", _Linear), ("up_skip", _Linear),
                ("pool_bn", _Bn), ("up_bn", _Bn), ("up_skip_bn", _Bn)]


class _Net(ctypes.Structure):
    _fields_ = [("dtype", _i32), ("n_stages", _i32), ("decoder", _i32), ("stem_in", _i32), ("patch", _i32 * levels.MAX_LEVELS),
                ("max_pair_density", _f32), ("reserved", _f32), ("stem_w", _ptr), ("stem_bn", _Bn), ("stage", _Stage * levels.MAX_LEVELS)]


class _Refresh(ctypes.Structure):
    _fields_ = [("dtype", _i32), ("n_cast", _i32), ("n_conv", _i32), ("n_mlp", _i32), ("cast_blocks", _i64),
                ("conv_blocks", _i64), ("mlp_blocks", _i64), ("cast", _ptr), ("conv", _ptr), ("mlp", _ptr),
                ("stem_src", _ptr), ("stem_dst", _ptr), ("stem_rows", _i64), ("stem_in", _i32), ("stem_padded", _i32)]


class Unsupported(Exception):
    """The model is not one the native forward covers."""


def _need(ok, why):
    if not ok:
        raise Unsupported(why)


CHANNELS = (32, 64, 128, 256, 512)
CONV_PACKED = (32, 64, 128)     # widths whose convolutions may take a tile form

# keys a caller may have put on the input that stand for work this path would do itself
_OWN_KEYS = ("serialized_code", "serialized_order", "serialized_inverse", "serialized_depth", "sparse_shape",
             "sparse_conv_feat", "pad", "unpad", "cu_seqlens_key", "pooling_inverse", "pooling_parent")


# what the native paths read of a module besides its children, parameters and buffers, once, when the model is described
# (a BatchNorm's momentum, a DropPath's rate and the orders are read at every forward)
_READ = {
    nn.GELU: ("approximate",), nn.Dropout: ("p",),
    nn.BatchNorm1d: ("eps", "num_features", "track_running_stats"), LayerNorm: ("eps", "normalized_shape"),
    SubMConv3d: ("kernel_size", "in_channels", "out_channels"), Block: ("channels", "pre_norm"),
    SerializedAttention: ("channels", "num_heads", "scale", "order_index", "patch_size", "enable_flash", "enable_rpe", "attn_drop"),
    SerializedPooling: ("stride", "reduce", "shuffle_orders", "traceable"), SerializedUnpooling: ("traceable",),
}
_PLAIN = (bool, int, float, str, tuple)
_shape = operator.attrgetter("shape")


# the classes a covered model is made of, with what they do
_FORWARDS = [(t, t.forward) for t in (
    nn.Linear, nn.GELU, nn.Dropout, nn.BatchNorm1d, nn.Identity, LayerNorm, SubMConv3d, MLP, Block, DropPath, Embedding, PointSequential,
    SerializedAttention, SerializedPooling, SerializedUnpooling)]


def _as_imported():
    return all(t.forward is f for t, f in _FORWARDS)


def _names(m):
    """What _READ names of a module."""
    names = _READ.get(type(m), ())
    if type(m) is SerializedAttention and not m.__dict__.get("enable_flash"):
        names = tuple(n for n in names if n != "patch_size")   # such a layer sets it at every forward
    return names


def _n_orders(attributes):
    orders = attributes.get("order")
    return len(orders) if isinstance(orders, (list, tuple)) else 0


def _values(dicts):
    return itertools.chain.from_iterable(map(dict.values, dicts))


def _same_objects(a, b):
    return len(a) == len(b) and all(map(operator.is_, a, b))


class Structure:
    """What of a model's modules the native paths rely on, and whether it still holds: which modules there are, their
    classes' forward, the attributes that were read, each parameter and statistic with its place and geometry. A change in any of them
    makes the model be looked at anew. same() runs in front of every forward (a few hundred modules, 0.08 - 0.13 ms), so it
    is lists compared by mapped C functions.

    It looks at the backbone (embedding, enc, dec) only; what else a subclass holds runs outside this forward. It holds the
    backbone's modules but not the model, whose table of engines (_ENGINES) would otherwise keep it alive for good."""

    PARTS = ("embedding", "enc", "dec")

    def __init__(self, model):
        self.why = None     # why no model of this structure is covered, as far as it shows here
        roots = [model._modules.get(name) for name in self.PARTS]
        self.modules = [m for root in roots if root is not None for m in root.modules()]
        # an instance attribute in the place of a method: the model does something else than its classes say
        if any(callable(getattr(type(m), name, None)) for m in self.modules for name in m.__dict__):
            self.why = "a method was replaced"
        self.hooks = [d for m in (model, *self.modules) for d in (m._forward_hooks, m._forward_pre_hooks, m._backward_hooks,
                                                                  m._backward_pre_hooks)]
        self.density = SubMConv3d.PAIR_MODE_MAX_DENSITY
        self._attributes = model.__dict__
        self._n_orders = _n_orders(model.__dict__)
        if not self._n_orders:
            self.why = "orders that are no list"
        if not _as_imported():
            self.why = "a class's forward was replaced"
        self._roots = [(model._modules, name, root) for name, root in zip(self.PARTS, roots) if root is not None]
        self._holders = [m._modules for m in self.modules if m._modules]
        self._children = list(_values(self._holders))
        # an instance attribute (a replaced forward) that came or went
        self._dicts = [m.__dict__ for m in self.modules]
        self._sizes = list(map(len, self._dicts))
        self._reads, self._values = [], []
        reads = [(m.__dict__, _names(m)) for m in self.modules] + [(model.__dict__, ("num_stages", "stride", "cls_mode"))]
        for attributes, names in reads:
            if not names:
                continue
            getter = operator.itemgetter(*names)
            try:
                values = getter(attributes)
            except KeyError as e:
                self.why = f"no attribute {e}"
                continue
            if not all(isinstance(v, _PLAIN) for v in (values if type(values) is tuple else (values,))):
                self.why = "an attribute that is no plain value"
                continue
            self._reads.append((getter, attributes))
            self._values.append(values)
        norms = [m for m in self.modules if isinstance(m, nn.BatchNorm1d)]
        self._tables = [m._parameters for m in self.modules if m._parameters] + [m._buffers for m in norms]
        self._held = list(_values(self._tables))
        counters = {id(m._buffers.get("num_batches_tracked")) for m in norms}
        self.tensors = [t for t in self._held if t is not None and id(t) not in counters]
        self._matrices = [t for t in self.tensors if t.dim() > 1]
        self._square = [t for t in self._matrices if t.dim() == 2 and t.shape[0] == t.shape[1]]
        self._places = self._places_now()
        # modules whose training flag changes what they compute
        self.flagged = [m for m in self.modules if isinstance(m, (nn.BatchNorm1d, nn.Dropout, DropPath, SerializedAttention))]

    def _places_now(self):
        # the same address with another shape is another weight too, and a square matrix may lie there transposed
        return [list(map(torch.Tensor.data_ptr, self.tensors)), list(map(_shape, self._matrices)), list(map(torch.Tensor.stride, self._square))]

    def hooked(self):
        hooks = torch.nn.modules.module
        return bool(hooks._global_forward_hooks or hooks._global_forward_pre_hooks or hooks._global_backward_hooks
                    or hooks._global_backward_pre_hooks or any(self.hooks))

    def same(self):
        """Whether everything this was made from still is what it was."""
        try:
            return (list(map(len, self._dicts)) == self._sizes and _as_imported()
                    and _n_orders(self._attributes) == self._n_orders and SubMConv3d.PAIR_MODE_MAX_DENSITY == self.density
                    and all(d.get(name) is root for d, name, root in self._roots)
                    and list(_values(self._holders)) == self._children and [f(d) for f, d in self._reads] == self._values
                    and _same_objects(list(_values(self._tables)), self._held) and self._places_now() == self._places)
        except KeyError:   # something went that was there
            return False


def _child(m, name, kind, why):
    """The child module of that name, which has to be of exactly that type."""
    child = m._modules.get(name)
    _need(type(child) is kind, why)
    return child


def _sequence(m, name, kinds, why):
    """The children of the PointSequential of that name; kinds says of which types they are to be."""
    parts = list(_child(m, name, PointSequential, why)._modules.values())
    _need(len(parts) == len(kinds) and all(type(c) in (k if type(k) is tuple else (k,)) for c, k in zip(parts, kinds)), why)
    return parts


def _check_gelu(m):
    _need(m.approximate == "none", "activation")


def _check_conv(m, kernel_size, biased):
    _need(m.kernel_size == kernel_size and m.PAIR_MODE_MAX_DENSITY == SubMConv3d.PAIR_MODE_MAX_DENSITY and (m.bias is not None) == biased
          and tuple(m.weight.shape) == (m.out_channels, *[kernel_size] * 3, m.in_channels)
          and (m.bias is None or m.bias.shape == (m.out_channels,)), "convolution")


def _check_block(b, c, n_orders):
    _need(type(b) is Block and b.pre_norm and b.channels == c and c in CHANNELS, "Block")
    conv, _, ln = _sequence(b, "cpe", (SubMConv3d, nn.Linear, LayerNorm), "xCPE")
    norms = [*_sequence(b, "norm1", (LayerNorm,), "norm"), *_sequence(b, "norm2", (LayerNorm,), "norm")]
    _need(ln.eps == norms[0].eps, "norm")
    _check_conv(conv, 3, True)
    _need(conv.in_channels == conv.out_channels == c, "xCPE")
    attn = _child(b, "attn", SerializedAttention, "attention")
    _need(attn.enable_flash and not attn.enable_rpe and "rpe" not in attn._modules and attn.channels == c
          and 1 <= attn.num_heads <= c and c % attn.num_heads == 0 and 0 <= attn.order_index < n_orders and attn.patch_size >= 1, "attention")
    for name in ("qkv", "proj"):
        _child(attn, name, nn.Linear, "attention")
    _child(attn, "proj_drop", nn.Dropout, "attention")
    mlp, = _sequence(b, "mlp", (MLP,), "MLP")
    for name in ("fc1", "fc2"):
        _child(mlp, name, nn.Linear, "MLP")
    _child(mlp, "drop", nn.Dropout, "MLP")
    _check_gelu(_child(mlp, "act", nn.GELU, "MLP"))
    _sequence(b, "drop_path", ((DropPath, nn.Identity),), "stochastic depth")


class Parts:
    """The modules of a model of the default architecture, stage by stage; Unsupported for any other."""

    class Stage:
        down = up = None
        enc = dec = ()
        bn = None            # of the pooling
        channels = dec_channels = patch = 0

    def __init__(self, model):
        S = model.num_stages
        self.n_orders = _n_orders(model.__dict__)
        _need(2 <= S <= levels.MAX_LEVELS and 1 <= self.n_orders <= levels.MAX_ORDERS and len(model.stride) == S - 1, "stages")
        embedding, enc = _child(model, "embedding", Embedding, "stem"), _child(model, "enc", PointSequential, "encoder")
        self.stem_conv, self.stem_bn, act = _sequence(embedding, "stem", (SubMConv3d, nn.BatchNorm1d, nn.GELU), "stem")
        _check_conv(self.stem_conv, 5, False)
        _check_gelu(act)
        _need(list(enc._modules) == [f"enc{s}" for s in range(S)], "encoder")
        dec = None if model.cls_mode else _child(model, "dec", PointSequential, "decoder")
        _need(dec is None or list(dec._modules) == [f"dec{s}" for s in reversed(range(S - 1))], "decoder")
        self.stages, below = [], self.stem_conv.out_channels
        for s in range(S):
            stage, st = _child(enc, f"enc{s}", PointSequential, "encoder stage"), Parts.Stage()
            st.enc = list(stage._modules.values())
            if s:
                _need(list(stage._modules)[:1] == ["down"] and type(st.enc[0]) is SerializedPooling, "pooling")
                st.down = st.enc.pop(0)
                st.bn, = _sequence(st.down, "norm", (nn.BatchNorm1d,), "pooling")
                act, = _sequence(st.down, "act", (nn.GELU,), "pooling")
                _check_gelu(act)
                _need(st.down.plan_kernel_sizes == (3,) and st.down.stride == model.stride[s - 1] and st.down.reduce in ops.REDUCE_OPS
                      and (not model.cls_mode or st.down.traceable)
                      and _child(st.down, "proj", nn.Linear, "pooling").in_features == below, "pooling")
                below = st.down.proj.out_features
            st.channels = below
            if dec is not None and s < S - 1:
                dstage = _child(dec, f"dec{s}", PointSequential, "decoder stage")
                st.dec = list(dstage._modules.values())
                _need(list(dstage._modules)[:1] == ["up"] and type(st.dec[0]) is SerializedUnpooling, "unpooling")
                st.up = st.dec.pop(0)
                _need(not st.up.traceable, "unpooling")
                kinds = nn.Linear, nn.BatchNorm1d, nn.GELU
                up, skip = _sequence(st.up, "proj", kinds, "unpooling"), _sequence(st.up, "proj_skip", kinds, "unpooling")
                _check_gelu(up[2])
                _check_gelu(skip[2])
                st.dec_channels = skip[0].out_features
                _need(st.dec_channels in CHANNELS and up[0].out_features == st.dec_channels, "decoder width")
            _need(below in CHANNELS, "width")
            for bs, c in ((st.enc, st.channels), (st.dec, st.dec_channels)):
                for b in bs:
                    _check_block(b, c, self.n_orders)
            sizes = [b.attn.patch_size for b in (*st.enc, *st.dec)]
            # the tables of a level are made for the patch size of the first attention that reaches it
            st.patch = sizes[0] if sizes else 1024
            _need(all(v >= st.patch for v in sizes), "patch sizes that shrink from the encoder to the decoder")
            self.stages.append(st)
        if dec is not None:
            width = self.stages[S - 1].channels
            for s in reversed(range(S - 1)):
                _need(self.stages[s].up.proj[0].in_features == width, "decoder widths")
                width = self.stages[s].dec_channels

    def layout(self, model):
        both = [[*st.enc, *st.dec] for st in self.stages]
        return levels.Layout(self.n_orders, model.stride, [st.patch for st in self.stages],
                             [[b.attn.order_index for b in bs] for bs in both],
                             [[(b.channels, b.channels) for b in bs] for bs in both], True,
                             [st.down.shuffle_orders for st in self.stages[1:]], only_pads0=not model.cls_mode)

    def widths(self):
        """Per level, the channel counts of its 3x3x3 convolutions."""
        return [sorted({b.channels for b in (*st.enc, *st.dec)}) for st in self.stages]


def check_linear(m, cin=None, cout=None, bias=True):
    """That a Linear is what its attributes say, of the widths asked for."""
    _need(type(m) is nn.Linear and (m.bias is not None or not bias) and tuple(m.weight.shape) == (m.out_features, m.in_features)
          and (m.bias is None or tuple(m.bias.shape) == (m.out_features,)), "Linear")
    _need((cin is None or m.in_features == cin) and (cout is None or m.out_features == cout), "Linear shape")


def check_layer_norm(m, c):
    _need(type(m) is LayerNorm and tuple(m.normalized_shape) == (c,)
          and all(p is not None and tuple(p.shape) == (c,) for p in (m.weight, m.bias)), "LayerNorm")


def check_batch_norm(m, c):
    _need(type(m) is nn.BatchNorm1d and m.track_running_stats and m.num_features == c
          and all(p is not None and tuple(p.shape) == (c,) for p in (m.weight, m.bias, m.running_mean, m.running_var)), "BatchNorm1d")


def job_table(rows, dtype, device):
    """A job table of the batch kernels in device memory, or None when it is empty."""
    if not rows:
        return None
    return torch.frombuffer(bytearray(np.array(rows, dtype=dtype).tobytes()), dtype=torch.uint8).to(device)


def coordinates(point):
    """(grid_coord int32, offset int64, batch int64 or None), contiguous, from a Point fresh from the caller."""
    point._ensure_grid_coord()
    batch = point.get("batch")
    if "offset" not in point:
        point["offset"] = batch2offset(batch)
    return (point["grid_coord"].to(torch.int32).contiguous(), point["offset"].to(torch.int64).contiguous(),
            None if batch is None else batch.to(torch.int64).contiguous())


def fill_point(point, index, s, feat, patch):
    """The keys of a level that serialization, sparsify and the attention put on its Point."""
    v = index.levels[s]
    i64, i32 = torch.int64, torch.int32
    point["feat"] = feat
    if s == 0:
        point["serialized_code"], point["serialized_order"], point["serialized_inverse"] = index.code, index.order, index.inverse
        point["_grid_max_host"] = index.grid_max
    point["serialized_depth"] = v.depth
    point["_offset_host"] = index.level_offsets[s]
    point["_sparse_indices"] = indices = index.tensor(v.indices, (v.n, 4), i32, "tables" if s else "first")
    point["sparse_shape"] = shape = [g + 96 for g in point["_grid_max_host"]]
    point["sparse_conv_feat"] = SparseConvTensor(feat, indices, shape, len(index.level_offsets[s]))
    if v.pad:
        point["pad"], point["unpad"] = index.tensor(v.pad, (v.n_pad,), i64), index.tensor(v.unpad, (v.n,), i64)
    point["cu_seqlens_key"] = index.tensor(v.cu, (v.n_seq + 1,), i32)
    point["_pad_patch"] = patch


class Copies:
    """The weight copies of an engine in device memory. They go when the model does, or when it has to be described again:
    a stream other than the one they were made on has to be known to the allocator by then."""

    def __init__(self):
        self._keep, self._streams = [], set()

    def used_here(self):
        """The kernels about to be queued on the current stream read the copies."""
        handle = ops._stream()
        if handle not in self._streams:
            for t in self._keep:
                if isinstance(t, torch.Tensor):
                    t.record_stream(torch.cuda.current_stream(self.device))   # nothing where it is the one they were made on
            self._streams.add(handle)


class Engine(Copies):
    def __init__(self, model, dtype):
        super().__init__()
        self.structure = Structure(model)
        parts = Parts(model)
        self.dtype = dtype
        self.device = self.structure.tensors[0].device
        params = [t for t in self.structure.tensors if isinstance(t, nn.Parameter)]
        kinds = {p.dtype for p in params}
        _need(self.structure.why is None, self.structure.why)
        _need(kinds == {dtype} or (kinds == {torch.float32} and dtype != torch.float32), "weights of several dtypes")
        _need(all(p.is_cuda and p.device == self.device and p.is_contiguous() for p in self.structure.tensors), "placement")
        self._casts, self._cast_out, self._cast_at = {}, None, 0
        self._jobs_conv, self._jobs_mlp = [], []
        self._cast = kinds != {dtype}
        if self._cast:
            total = sum(-(-p.numel() // 128) * 128 for p in params)
            self._cast_out = torch.empty(total, dtype=dtype, device=self.device)
            self._keep.append(self._cast_out)
        self._describe(model, parts)
        self._finish_jobs()

    # ---- pointers -------------------------------------------------------------------------------------------------
    def _p(self, t):
        """Address of a parameter in the compute dtype: its own, or that of its copy (casts)."""
        if t is None:
            return None
        if not self._cast:
            return t.data_ptr()
        held = self._casts.get(t)
        if held is None:
            held = self._casts[t] = self._cast_out.data_ptr() + self._cast_at * self._cast_out.element_size()
            self._cast_at += -(-t.numel() // 128) * 128
        return held

    def _linear(self, m, cin=None, cout=None, bias=True):
        check_linear(m, cin, cout, bias)
        return _Linear(self._p(m.weight), self._p(m.bias), m.in_features, m.out_features)

    def _norm(self, m, c):
        check_layer_norm(m, c)
        return _Norm(self._p(m.weight), self._p(m.bias), m.eps, 0)

    def _bn(self, m, c):
        check_batch_norm(m, c)
        stats = m.running_mean.dtype
        _need(m.running_var.dtype == stats and stats in (torch.float32, self.dtype), "BatchNorm1d statistics")
        return _Bn(m.running_mean.data_ptr(), m.running_var.data_ptr(), self._p(m.weight), self._p(m.bias), m.eps,
                   int(stats == torch.float32))

    def _packed(self, elements):
        t = torch.empty(elements, dtype=self.dtype, device=self.device)
        self._keep.append(t)
        return t.data_ptr()

    def _block(self, b, c):
        conv, lin, attn, mlp = b.cpe[0], b.cpe[1], b.attn, b.mlp[0]
        d = _Block(channels=c, heads=attn.num_heads, row=attn.order_index, scale=attn.scale)
        d.conv_w, d.conv_b = self._p(conv.weight), self._p(conv.bias)
        d.cpe, d.qkv, d.proj = self._linear(lin, c, c), self._linear(attn.qkv, c, 3 * c), self._linear(attn.proj, c, c)
        d.fc1, d.fc2 = self._linear(mlp.fc1, c, 4 * c), self._linear(mlp.fc2, 4 * c, c)
        d.ln_cpe, d.ln1, d.ln2 = self._norm(b.cpe[2], c), self._norm(b.norm1[0], c), self._norm(b.norm2[0], c)
        if self.dtype != torch.float32:
            if c in CONV_PACKED:
                d.conv_packed = self._packed(27 * c * c)
                self._jobs_conv.append((d.conv_w, d.conv_packed, c, 27))
            if c >= 128:
                d.mlp_packed = self._packed(8 * c * c)
                self._jobs_mlp.append((d.fc1.w, d.fc2.w, d.mlp_packed, c, 0))
            if c in (128, 256):
                d.proj_packed = self._packed(c * c)
                self._jobs_mlp.append((d.proj.w, 0, d.proj_packed, c, 1))
                d.head_packed = self._packed(4 * c * c)
                self._jobs_mlp.append((d.cpe.w, 0, d.head_packed, c, 1))
                self._jobs_mlp.append((d.qkv.w, 0, d.head_packed + c * c * 2, c, 3))
        return d

    def _describe(self, model, p):
        """ptv3_net of the model, p its Parts; Unsupported where it is not the default architecture."""
        net = self.net = _Net(dtype=ops.DTYPE_CODES[self.dtype], n_stages=len(p.stages), decoder=int(not model.cls_mode))
        net.stem_in, net.max_pair_density = p.stem_conv.in_channels, self.structure.density
        net.stem_w = self._p(p.stem_conv.weight)
        net.stem_bn = self._bn(p.stem_bn, p.stem_conv.out_channels)
        self._refresh = r = _Refresh(dtype=net.dtype)
        if self.dtype != torch.float32:
            padded = -(-p.stem_conv.in_channels // 16) * 16
            r.stem_rows, r.stem_in, r.stem_padded = p.stem_conv.out_channels * 125, p.stem_conv.in_channels, padded
            r.stem_src = net.stem_w
            r.stem_dst = net.stem_w = self._packed(r.stem_rows * padded)
        for s, st in enumerate(p.stages):
            d = net.stage[s]
            d.channels, d.n_enc, d.dec_channels, d.n_dec = st.channels, len(st.enc), st.dec_channels, len(st.dec)
            if st.down is not None:
                d.pool = self._linear(st.down.proj, None, st.channels)
                d.pool_bn, d.pool_reduce = self._bn(st.bn, st.channels), ops.REDUCE_OPS[st.down.reduce]
            if st.up is not None:
                d.up, d.up_skip = self._linear(st.up.proj[0]), self._linear(st.up.proj_skip[0], st.channels)
                d.up_bn, d.up_skip_bn = self._bn(st.up.proj[1], st.dec_channels), self._bn(st.up.proj_skip[1], st.dec_channels)
            for attr, bs, c in (("enc", st.enc, st.channels), ("dec", st.dec, st.dec_channels)):
                if bs:
                    arr = (_Block * len(bs))(*[self._block(b, c) for b in bs])
                    self._keep.append(arr)
                    setattr(d, attr, ctypes.addressof(arr))
            net.patch[s] = st.patch
        self.out_channels = p.stages[0].dec_channels or None
        self.layout = p.layout(model)
        half = self.dtype != torch.float32
        form = _lib.load().ptv3_conv_form
        widths = p.widths()

        def want(level, v):
            flags = levels.PAIRS5 if level == 0 else 0
            for c in widths[level]:
                flags |= levels.TILES if half and form(v.n, v.n_pairs, c) else levels.PAIRS
            return flags

        self.want = want

    def _finish_jobs(self):
        lib, r = _lib.load(), self._refresh

        def table(rows, dtype):
            t = job_table(rows, dtype, self.device)
            self._keep.append(t)
            return t.data_ptr() if t is not None else None

        rows, at = [], 0
        for t, dst in self._casts.items():
            rows.append((t.data_ptr(), dst, 1, 1, t.numel(), 0, at))
            at += lib.ptv3_cast_params_blocks(1, 1, t.numel(), 0)
        r.cast, r.n_cast, r.cast_blocks = table(rows, ops._CAST_JOB), len(rows), at
        rows, at = [], 0
        for src, dst, c, taps in self._jobs_conv:
            rows.append((src, dst, c, taps, at))
            at += lib.ptv3_subm_conv_pack_weight_blocks(c, taps)
        r.conv, r.n_conv, r.conv_blocks = table(rows, ops._PACK_JOB), len(rows), at
        rows, at = [], 0
        for w1, w2, dst, c, k in self._jobs_mlp:
            rows.append((w1, w2, dst, c, k, at))
            at += k * lib.ptv3_linear_pack_weights_blocks(c) if k else lib.ptv3_mlp_pack_weights_blocks(c)
        r.mlp, r.n_mlp, r.mlp_blocks = table(rows, ops._MLP_PACK_JOB), len(rows), at

    # ---- one forward ----------------------------------------------------------------------------------------------
    def forward(self, model, data):
        """The Point that PointTransformerV3.forward returns for these inputs (see Inputs in `accepts`)."""
        lib = _lib.load()
        feat = data["feat"].contiguous()
        point = Point.__new__(Point)
        dict.update(point, data)
        self.used_here()

        def refresh():
            # whoever writes the parameters behind autograd's back leaves no trace on them: every derived copy is
            # redone once per forward
            _lib.check(lib.ptv3_net_refresh(ctypes.byref(self._refresh), ops._stream()), "ptv3_net_refresh")

        def index_of(between=None):
            return levels.build(self.layout, *coordinates(point), list(model.order), model.shuffle_orders, self.want, between=between)

        if model.overlap_index_prologue:
            if model._prologue_state is None or model._prologue_state.device != feat.device:
                model._prologue_state = ops.PrologueOverlap(feat.device)
            refresh()
            with model._prologue_state.scope():
                # the conversions of the inputs too: that stream waits for nothing, so what it reads is made on it
                index = index_of()
        else:
            model._prologue_state = None
            index = index_of(between=refresh)
        lv = index.levels
        n = feat.shape[0]
        stage_out, rows = None, None
        if model.cls_mode:
            rows = [torch.empty((lv[s].n, self.net.stage[s].channels), dtype=self.dtype, device=feat.device)
                    for s in range(self.net.n_stages)]
            stage_out = (_ptr * len(rows))(*[t.data_ptr() for t in rows])
            out = rows[-1]
        else:
            out = torch.empty((n, self.out_channels), dtype=self.dtype, device=feat.device)
        nbytes = lib.ptv3_features_bytes(ctypes.byref(self.net), lv, stage_out)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=feat.device)
        _lib.check(lib.ptv3_features_fwd(ctypes.byref(self.net), lv, feat.data_ptr(), ops.DTYPE_CODES[feat.dtype], stage_out,
                                         None if model.cls_mode else out.data_ptr(), ws.data_ptr(), nbytes, ops._stream()),
                   "ptv3_features_fwd")
        point["batch"] = index.batch
        fill_point(point, index, 0, rows[0] if model.cls_mode else out, self.net.patch[0])
        if model.cls_mode:
            for s in range(1, len(rows)):
                point = self._pooled(point, index, s, rows[s])
        if model._prologue_state is not None:
            model._prologue_state.forward_queued(point)
        return point

    def _pooled(self, parent, index, s, feat):
        v, k = index.levels[s], index.n_orders
        i64 = torch.int64
        idx_ptr = index.tensor(v.idx_ptr, (v.n + 1,), i64)
        members = parent["serialized_order"][0]
        shift = parent["serialized_depth"] - v.depth
        point = Point.__new__(Point)
        if "coord" in parent:
            point["coord"] = ops.segment_reduce(parent["coord"].float(), members, idx_ptr, "mean")
        dict.update(
            point, grid_coord=index.tensor(v.grid, (v.n, 3), torch.int32), serialized_code=index.tensor(v.code, (k, v.n), i64),
            serialized_order=index.tensor(v.order, (k, v.n), i64), serialized_inverse=index.tensor(v.inverse, (k, v.n), i64),
            batch=index.tensor(v.batch, (v.n,), i64),
            offset=index.tensor(v.offset, (len(index.level_offsets[s]),), i64, "first"), _pool_members=(members, idx_ptr),
            _grid_max_host=[g >> shift for g in parent["_grid_max_host"]],
            pooling_inverse=index.tensor(v.cluster, (index.levels[s - 1].n,), i64), pooling_parent=parent)
        for key in ("condition", "context"):
            if key in parent:
                point[key] = parent[key]
        fill_point(point, index, s, feat, self.net.patch[s])
        return point


# model -> {(compute dtype, encoder only): Engine or Refused}; neither holds the model, so it goes when its user lets it go
_ENGINES = weakref.WeakKeyDictionary()


def _compute_dtype(feat, weight):
    """The dtype the model's rows would have, or None where the modules mix dtypes."""
    if torch.is_autocast_enabled():
        dt = torch.get_autocast_dtype("cuda")
        return dt if weight.dtype in (torch.float32, dt) and dt != torch.float32 else None
    return feat.dtype if feat.dtype == weight.dtype else None


def plain_inputs(data):
    """Whether `data` is what a caller hands to a forward and nothing a forward would have made itself: features and
    coordinates on the GPU, scene ends or ids, no tables."""
    if type(data) not in (dict, AttrDict, Point) or ops._LAUNCH_TIMER is not None or ops.Readback.blocking:
        return False
    feat = data.get("feat")
    if not isinstance(feat, torch.Tensor) or not feat.is_cuda or feat.dim() != 2 or feat.shape[0] < 1 or feat.dtype not in ops.DTYPE_CODES:
        return False
    if any(k in data for k in _OWN_KEYS) or any(k.startswith("_") for k in data) or not ("offset" in data or "batch" in data):
        return False
    n, where, offset, batch = feat.shape[0], data.get("grid_coord", data.get("coord")), data.get("offset"), data.get("batch")
    # the kernels take addresses: what is not of these shapes on this GPU is the modules' to convert or to refuse
    return (_placed(where, feat, 2) and where.shape == (n, 3) and ("grid_coord" in data or "grid_size" in data)
            and ("offset" not in data or (_placed(offset, feat, 1) and offset.shape[0] > 0))
            and ("batch" not in data or (_placed(batch, feat, 1) and batch.shape[0] == n)))


def _placed(t, feat, dim):
    return isinstance(t, torch.Tensor) and t.device == feat.device and t.dim() == dim


def _stem_weight(model):
    """The weight of the stem's convolution, or None where the model has another embedding."""
    conv = model._modules.get("embedding")
    for name in ("stem", "conv"):
        conv = None if conv is None else conv._modules.get(name)
    return conv.weight if type(conv) is SubMConv3d else None


def engine_for(model, data):
    """The Engine that computes model(data), or None: the modules do."""
    if model.training or torch.is_grad_enabled() or not plain_inputs(data):
        return None
    feat = data["feat"]
    weight = _stem_weight(model)
    dtype = None if weight is None or weight.device != feat.device else _compute_dtype(feat, weight)
    if dtype not in ops.DTYPE_CODES or feat.shape[1] != weight.shape[-1]:
        return None
    held = _ENGINES.setdefault(model, {})
    key = (dtype, model.cls_mode)
    engine = held.get(key)
    if engine is None or not engine.structure.same():
        try:
            engine = Engine(model, dtype)
        except Unsupported as e:
            engine = Refused(model, str(e))
        held[key] = engine
    if isinstance(engine, Refused) or engine.structure.hooked() or any(m.training for m in engine.structure.flagged):
        return None
    return engine


class Refused:
    """A model the native paths do not cover, remembered until its structure or weights move."""

    def __init__(self, model, why):
        self.why, self.structure = why, Structure(model)
