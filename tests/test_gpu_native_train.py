"""The natively queued training step against the same model's modules: rows, running statistics, every gradient."""
import copy

import numpy as np
import pytest
import torch

from gpu_util import DEV
from test_gpu_native import KW, _inputs

pytestmark = pytest.mark.gpu


def _step(model, data, dtype, use, monkeypatch, seed=11):
    from pointtransformerv3_amd import native_train
    taken, real = [], native_train.engine_for
    monkeypatch.setattr(native_train, "engine_for",
                        (lambda m, d: taken.append(real(m, d)) or taken[-1]) if use else (lambda m, d: None))
    model.zero_grad(set_to_none=True)
    torch.manual_seed(seed)
    with torch.autocast("cuda", dtype=dtype):
        point = model(dict(data))
    g = torch.Generator(device=DEV).manual_seed(1)
    # a coherent gradient (few classes, by place): a sum of independent signs would amplify every rounding
    label = (data["grid_coord"].sum(1) % 5).long()
    w = torch.randn(5, point.feat.shape[1], generator=g, device=DEV)
    point.feat.backward((w[label] * 0.05).to(point.feat.dtype))
    monkeypatch.setattr(native_train, "engine_for", real)
    assert not use or taken[0] is not None, "the native path was not taken"
    return point


def _compare(model, data, dtype, monkeypatch, tol):
    other = copy.deepcopy(model)
    a, b = _step(model, data, dtype, True, monkeypatch), _step(other, data, dtype, False, monkeypatch)
    assert a.feat.dtype == b.feat.dtype == torch.float32
    rel = lambda x, y: float((x.double() - y.double()).norm() / y.double().norm().clamp_min(1e-30))
    errs = {"feat": rel(a.feat.detach(), b.feat.detach())}
    for (name, p), q in zip(model.named_parameters(), other.parameters()):
        assert p.grad.shape == q.grad.shape and torch.isfinite(p.grad).all(), name
        errs[name] = rel(p.grad, q.grad)
    bufs = [(n, x, y) for (n, x), y in zip(model.named_buffers(), other.buffers())]
    for n, x, y in bufs:
        assert torch.equal(x, y) if not x.is_floating_point() else rel(x, y) < tol, (n, rel(x, y))
    for key in ("batch", "serialized_order", "pad", "unpad", "cu_seqlens_key"):
        assert torch.equal(a[key], b[key])
    flat = lambda m: torch.cat([p.grad.reshape(-1) for p in m.parameters()])
    assert rel(flat(model), flat(other)) < tol, sorted(errs.items(), key=lambda kv: -kv[1])[:5]
    ranked = sorted(errs.values())
    assert ranked[len(ranked) // 2] < tol, ranked[len(ranked) // 2]
    return errs


@pytest.mark.parametrize("sizes", [(6000,), (9000, 150, 4000)])
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-2), (torch.bfloat16, 6e-2)])
def test_native_training_step_matches_the_modules(dtype, tol, sizes, monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(**dict(KW, enc_depths=(1, 2, 2, 1, 1))).to(DEV).train()
    _compare(model, _inputs(4, sizes, torch.float32), dtype, monkeypatch, tol)


def test_native_training_step_without_stochastic_depth_and_with_frozen_parameters(monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    data = _inputs(4, (7000,), torch.float32)
    _compare(model, data, torch.float16, monkeypatch, 2e-2)
    model.enc.enc2.requires_grad_(False)
    _step(model, data, torch.float16, True, monkeypatch)
    assert all((p.grad is None) == n.startswith("enc.enc2.") for n, p in model.named_parameters())


def test_native_training_follows_the_optimizer_and_leaves_other_modes_alone(monkeypatch):
    from pointtransformerv3_amd import PointTransformerV3, native_train
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    data = _inputs(4, (5000,), torch.float32)
    opt = torch.optim.AdamW(model.parameters(), lr=1e-3, fused=True)
    for _ in range(2):
        _step(model, data, torch.bfloat16, True, monkeypatch)
        opt.step()
    _compare(model, data, torch.bfloat16, monkeypatch, 6e-2)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert native_train.engine_for(model, data) is not None
        model.enc.enc1.down.norm[0].eval()                       # a frozen BatchNorm: the modules
        assert native_train.engine_for(model, data) is None
        model.train()
        assert native_train.engine_for(model, dict(data, feat=data["feat"].clone().requires_grad_())) is None
        with torch.no_grad():
            assert native_train.engine_for(model, data) is None
    assert native_train.engine_for(model, data) is None          # no autocast: the modules
    # a second backward over a step whose graph was freed fails as any other does
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = model(dict(data)).feat
    out.sum().backward()
    with pytest.raises(RuntimeError):
        out.sum().backward()


@pytest.mark.parametrize("how", ["checkpoint", "offload"])
def test_native_training_step_under_saved_tensor_hooks(how):
    """What autograd keeps for the backward may be recomputed or moved: stochastic-depth factors and activations are read
    from where they are when the backward runs. The same step twice: the batch statistics are summed by atomics, so single
    roundings to half differ as they do between this path and the modules, whose tolerance is taken; another set of rows
    kept by stochastic depth, or activations overwritten, would be wrong by the size of a branch."""
    from torch.utils.checkpoint import checkpoint
    from pointtransformerv3_amd import PointTransformerV3, native_train
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).to(DEV).train()
    data = _inputs(4, (6000,), torch.float32)
    taken, real = [], native_train.engine_for

    def step(hooked):
        model.zero_grad(set_to_none=True)
        torch.manual_seed(5)
        with torch.autocast("cuda", dtype=torch.float16):
            if hooked and how == "checkpoint":
                feat = checkpoint(lambda d: model(dict(d)).feat, data, use_reentrant=False)
            elif hooked:
                with torch.autograd.graph.save_on_cpu():
                    feat = model(dict(data)).feat
            else:
                feat = model(dict(data)).feat
        # other work takes the memory that was let go
        fill = [torch.full((1 << k,), float("nan"), device=DEV) for k in range(6, 22)]
        del fill
        feat.backward(torch.full_like(feat, 0.01))
        return feat.detach().clone(), [p.grad.clone() for p in model.parameters()]

    native_train.engine_for = lambda m, d: taken.append(real(m, d)) or taken[-1]
    try:
        want, got = step(False), step(True)
    finally:
        native_train.engine_for = real
    assert len(taken) >= 2 and all(e is not None for e in taken)
    rel = lambda x, y: float((x.double() - y.double()).norm() / y.double().norm())
    assert rel(got[0], want[0]) < 2e-2
    assert rel(*(torch.cat([g.reshape(-1) for g in gs]) for gs in (got[1], want[1]))) < 2e-2


def test_native_training_step_notices_weights_written_before_its_backward():
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    data = _inputs(4, (3000,), torch.float32)
    step = lambda: model(dict(data)).feat
    with torch.autocast("cuda", dtype=torch.bfloat16):
        first = step()
        with torch.no_grad():
            model.enc.enc2.block0.attn.proj.weight.mul_(1.5)
            model.enc.enc2.block0.attn.proj.bias.mul_(1.5)
        second = step()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        first.sum().backward()
    second.sum().backward()
    assert all(torch.isfinite(p.grad).all() for p in model.parameters())


@pytest.mark.parametrize("extra", ["head", "mask token", "shared block", "shared norm"])
def test_gradients_of_models_that_hold_more_or_less_than_the_backbone(extra, monkeypatch):
    """A parameter outside the backbone gets its own gradient and nothing else; one used twice gets the sum of both."""
    from pointtransformerv3_amd import PointTransformerV3, native_train

    class Segmentor(PointTransformerV3):
        def __init__(self, **kw):
            super().__init__(**kw)
            if extra == "head":
                self.head = torch.nn.Linear(64, 13)
            elif extra == "mask token":
                self.token = torch.nn.Parameter(torch.ones(64))

        def forward(self, data):
            point = super().forward(data)
            if extra == "head":
                point.feat = self.head(point.feat)
            elif extra == "mask token":
                point.feat = point.feat * self.token
            return point

    torch.manual_seed(3)
    model = Segmentor(drop_path=0.0, **dict(KW, enc_depths=(1, 2, 2, 1, 1))).to(DEV).train()
    if extra == "shared block":
        model.enc.enc1.block1 = model.enc.enc1.block0
    elif extra == "shared norm":
        model.enc.enc2.block1.norm2 = model.enc.enc2.block0.norm1
    data = _inputs(4, (5000,), torch.float32)
    other = copy.deepcopy(model)
    label = (data["grid_coord"].sum(1) % 5).long()
    taken, real = [], native_train.engine_for

    def grads(m, use):
        monkeypatch.setattr(native_train, "engine_for", (lambda a, b: taken.append(real(a, b)) or taken[-1]) if use else lambda a, b: None)
        torch.full((1 << 24,), float("nan"), device=DEV)     # what freed memory holds
        torch.manual_seed(5)
        with torch.autocast("cuda", dtype=torch.float16):
            feat = m(dict(data)).feat
        w = torch.randn(5, feat.shape[1], generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
        feat.backward((w[label] * 0.05).to(feat.dtype))
        return {n: p.grad for n, p in m.named_parameters()}

    got, want = grads(model, True), grads(other, False)
    assert (taken[0] is None) == extra.startswith("shared")
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))
    assert set(got) == set(want) and all(torch.isfinite(g).all() for g in got.values())
    errs = {n: rel(got[n], want[n]) for n in want}
    assert rel(torch.cat([got[n].flatten() for n in want]), torch.cat([want[n].flatten() for n in want])) < 2e-2, errs
    for n in ("head.weight", "head.bias", "token"):
        assert errs.get(n, 0.0) < 2e-2, errs


def test_native_training_step_follows_a_momentum_schedule(monkeypatch):
    """Running statistics after steps whose BatchNorm momentum changes in between (and is None in the last)."""
    from pointtransformerv3_amd import PointTransformerV3, native_train
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    other = copy.deepcopy(model)
    data = _inputs(4, (3000,), torch.float32)
    for i, momentum in enumerate((0.01, 0.5, 0.2)):
        for m, use in ((model, True), (other, False)):
            for bn in m.modules():
                if isinstance(bn, torch.nn.BatchNorm1d):
                    bn.momentum = momentum
            _step(m, data, torch.float16, use, monkeypatch)
        for (n, x), y in zip(model.named_buffers(), other.buffers()):
            assert torch.allclose(x.float(), y.float(), rtol=2e-2, atol=2e-2 * float(y.float().abs().max())), (i, n)
    model.enc.enc1.down.norm[0].momentum = None
    with torch.autocast("cuda", dtype=torch.float16):
        assert native_train.engine_for(model, data) is None


@pytest.mark.parametrize("extent", [18, 32])
def test_native_training_step_in_dense_volumes(extent, monkeypatch):
    """Float rows in the small volume, the neighbour map in the large one: forward and input gradients as the modules'."""
    from pointtransformerv3_amd import PointTransformerV3
    from test_gpu_native import _volume
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    _compare(model, _volume(extent, torch.float32), torch.float16, monkeypatch, 2e-2)


def test_native_training_step_on_a_second_stream(monkeypatch):
    """A step on a stream of its own after one on the default stream: the same rows and gradients."""
    from pointtransformerv3_amd import PointTransformerV3
    torch.manual_seed(3)
    model = PointTransformerV3(drop_path=0.0, **KW).to(DEV).train()
    data = _inputs(4, (5000,), torch.float32)
    first = _step(model, data, torch.float16, True, monkeypatch).feat.detach().clone()
    want = torch.cat([p.grad.reshape(-1) for p in model.parameters()])
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(3):
            point = _step(model, data, torch.float16, True, monkeypatch)
        got = torch.cat([p.grad.reshape(-1) for p in model.parameters()])
    side.synchronize()
    rel = lambda x, y: float((x.double() - y.double()).norm() / y.double().norm())
    # batch statistics are summed by atomics: single roundings to half differ
    assert rel(point.feat.detach(), first) < 2e-2 and rel(got, want) < 2e-2


@pytest.mark.parametrize("sizes", [(300,), (2000, 900), (30_000, 12_000)])
@pytest.mark.parametrize("caller", ["default stream", "another stream"])
def test_weight_gradients_beside_the_backward_are_those_of_one_stream(sizes, caller, monkeypatch):
    """From one group of weight gradients to several that take turns in the two arenas, twice over one forward's activations.
    An operand overwritten too early makes a parameter's gradient wrong by its own size, so every parameter is held by itself.
    The backward's sums by atomics enter its chain at the first BatchNorm: the matrices of the blocks before it have the same
    bits. From there on single roundings to half differ from run to run, on one stream as on two: 2.4 % of a parameter's norm
    were seen (the first block's norm of 300 voxels), 5 % are allowed. A bias in front of a BatchNorm has no gradient but
    rounding, up to 3.3e-4 of that of its layer's weight were seen, where the other biases have 8e-3 and more: 1e-3."""
    from pointtransformerv3_amd import PointTransformerV3, native_train
    torch.manual_seed(3)
    model = PointTransformerV3(**KW).to(DEV).train()
    data = _inputs(4, sizes, torch.float32)
    on = torch.cuda.Stream() if caller == "another stream" else torch.cuda.current_stream()
    on.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(on):
        _step(model, data, torch.float16, True, monkeypatch)
        engine = native_train._ENGINES[model][torch.float16]
        assert engine.net.side and engine.net.side != on.cuda_stream
        with torch.autocast("cuda", dtype=torch.float16):
            feat = model(dict(data)).feat
        runs = {"one stream": [], "second stream": [], "the caller's stream": []}
        beside = engine.side.cuda_stream
        for name, side in (("second stream", beside), ("one stream", None), ("the caller's stream", on.cuda_stream), ("second stream", beside)):
            engine.net.side = side
            model.zero_grad(set_to_none=True)
            feat.backward(torch.full_like(feat, 0.01), retain_graph=True)
            runs[name].append([p.grad.double() for p in model.parameters()])
    torch.cuda.synchronize()
    (alone,) = runs.pop("one stream")
    names = [name for name, _ in model.named_parameters()]
    for i, name in enumerate(names):
        allowed = 5e-2 * float(alone[i].norm())
        if name.endswith(".bias"):
            allowed += 1e-3 * float(alone[names.index(name[:-4] + "weight")].norm())
        same = name.startswith("dec.dec0.block") and any(part in name for part in ("cpe.0", "cpe.1", "attn", "mlp"))
        for case, got in ((c, g[i]) for c, gs in runs.items() for g in gs):
            assert torch.isfinite(got).all(), (name, case)
            assert torch.equal(got, alone[i]) if same else float((got - alone[i]).norm()) <= allowed, (name, case)
    for got in (g for gs in runs.values() for g in gs):
        got, want = torch.cat([g.reshape(-1) for g in got]), torch.cat([g.reshape(-1) for g in alone])
        assert float((got - want).norm() / want.norm()) < 2e-2
