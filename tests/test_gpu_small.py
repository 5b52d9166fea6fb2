"""Forms that only small inputs take: long segments of few, the pair form of 64- and 128-channel convolutions."""
import pytest
import torch

from gpu_util import DEV, rel_err, to_dev, unique_voxels
from oracle import functional as OF
from oracle import indexing as OI

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("reduce", ["max", "mean", "sum", "min"])
@pytest.mark.parametrize("lengths,c", [([700], 512), ([0, 900, 1, 255, 256, 257, 63, 0], 64), ([4000, 5], 8), ([300, 100], 136)])
def test_long_segments(lengths, c, reduce, dtype):
    from pointtransformerv3_amd import ops
    g = torch.Generator().manual_seed(sum(lengths) + c)
    n = sum(lengths)
    x = torch.randn(n, c, generator=g).to(dtype)
    at = torch.randperm(n, generator=g)
    ptr = torch.tensor([0] + lengths).cumsum(0)
    got = ops.segment_reduce(x.to(DEV), at.to(DEV), ptr.to(DEV), reduce)
    rows = x.float()[at]
    want = torch.zeros(len(lengths), c)
    for s in range(len(lengths)):
        part = rows[ptr[s]:ptr[s + 1]]
        if len(part):
            want[s] = {"max": part.amax(0), "min": part.amin(0), "mean": part.mean(0), "sum": part.sum(0)}[reduce]
    assert rel_err(got, want) < {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c,n,extent", [(64, 2000, 14), (64, 6000, 40), (128, 700, 10), (128, 7000, 24)])
def test_convolution_of_few_pairs(c, n, extent, dtype):
    import numpy as np

    from pointtransformerv3_amd import _lib, ops
    from pointtransformerv3_amd.sparse import SparseConvTensor, SubMConv3d
    grid, batch, _ = unique_voxels(np.random.default_rng(n), n, extent, nb=2)
    idx = np.concatenate([batch[:, None], grid], 1).astype(np.int32)
    torch.manual_seed(n)
    conv = SubMConv3d(c, c, 3, bias=True, indice_key="k").to(dtype).to(DEV).requires_grad_(False)
    x = torch.randn(len(grid), c).to(dtype)
    plan = ops.conv_plan_direct(to_dev(idx), 3)
    assert _lib.load().ptv3_conv_form(len(grid), plan.n_pairs, c) == 0
    got = conv(SparseConvTensor(x.to(DEV), to_dev(idx), [extent + 96] * 3, 2)).features
    want = OF.subm_conv(x.float(), OI.subm_kmap(idx), conv.weight.float().cpu(), conv.bias.float().cpu())
    assert rel_err(got, want) < {torch.float16: 2e-2, torch.bfloat16: 2e-2}[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c,n,extent", [(64, 1, 2), (64, 33, 4), (64, 2000, 14), (64, 6000, 40), (128, 1, 2), (128, 129, 8), (128, 700, 10), (128, 7000, 24)])
def test_convolution_of_few_pairs_rounds_once(c, n, extent, dtype):
    """The pair form with product rows in float against 64 bits: products exact in float, sums of at most 27 taps in float,
    one rounding to half, as in the tile form whose place it takes -- its error is the tile form's, not 1.1 times it."""
    import numpy as np

    from pointtransformerv3_amd import _lib, ops
    grid, batch, _ = unique_voxels(np.random.default_rng(n), n, extent, nb=2)
    idx = to_dev(np.concatenate([batch[:, None], grid], 1).astype(np.int32))
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(len(grid), c, generator=g, device=DEV).to(dtype)
    w = (torch.randn(c, 27, c, generator=g, device=DEV) / (27 * c) ** 0.5).to(dtype)
    bias = torch.randn(c, generator=g, device=DEV).to(dtype)
    plan = ops.conv_plan_direct(idx, 3)
    assert _lib.load().ptv3_conv_few_pairs(plan.n_pairs, c) and not _lib.load().ptv3_conv_few_pairs(plan.n_pairs, 32)
    want = bias.double().expand(len(grid), c).clone()
    nbr = ops.kmap_build(idx, 3).long()
    for t in range(27):
        on = nbr[:, t] >= 0
        want[on] += x.double()[nbr[on, t]] @ w[:, t].double().t()
    err = lambda y: float((y.double() - want).norm() / want.norm())
    wide = err(ops.subm_conv_pairs(x, plan, w, bias, wide=True))
    tile = err(ops.subm_conv_tiles(x, plan, ops.conv_pack_weight(w, 27, dtype), bias))
    eps = torch.finfo(dtype).eps
    assert wide <= 1.02 * tile + 0.02 * eps and wide < 0.5 * eps
    assert torch.equal(ops.subm_conv_pairs(x, plan, w, None, wide=True), ops.subm_conv_pairs(x, plan, w, torch.zeros_like(bias), wide=True))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ks,cin,cout,n,extent", [(3, 32, 32, 1700, 12), (3, 256, 256, 900, 10), (3, 512, 512, 500, 8), (5, 16, 32, 1000, 10),
                                                  (3, 16, 8, 65, 5), (3, 48, 40, 300, 8), (3, 128, 200, 300, 8), (3, 512, 64, 200, 7)])
def test_pair_form_with_float_rows_rounds_once(ks, cin, cout, n, extent, dtype):
    """The shapes that take it in small dense volumes, and the edges of what it takes, against 64 bits: below one rounding."""
    import numpy as np

    from pointtransformerv3_amd import ops
    grid, batch, _ = unique_voxels(np.random.default_rng(n), n, extent)
    idx = to_dev(np.concatenate([batch[:, None], grid], 1).astype(np.int32))
    g = torch.Generator(device=DEV).manual_seed(n)
    taps = ks ** 3
    x = torch.randn(n, cin, generator=g, device=DEV).to(dtype)
    w = (torch.randn(cout, taps, cin, generator=g, device=DEV) / (taps * cin) ** 0.5).to(dtype)
    bias = torch.randn(cout, generator=g, device=DEV).to(dtype)
    want = bias.double().expand(n, cout).clone()
    nbr = ops.kmap_build(idx, ks).long()
    for t in range(taps):
        on = nbr[:, t] >= 0
        want[on] += x.double()[nbr[on, t]] @ w[:, t].double().t()
    got = ops.subm_conv_pairs(x, ops.conv_plan_direct(idx, ks), w, bias, wide=True)
    assert float((got.double() - want).norm() / want.norm()) < 0.5 * torch.finfo(dtype).eps


def test_pair_form_with_float_rows_refuses_other_shapes():
    from pointtransformerv3_amd import _lib
    lib, x = _lib.load(), torch.zeros(64, device=DEV)
    call = lambda dt, cin, cout, taps=27: lib.ptv3_subm_conv_pairs_wide_fwd(x.data_ptr(), dt, 1, cin, taps, 0, x.data_ptr(), x.data_ptr(),
                                                                           0, 0, x.data_ptr(), 0, cout, 0, x.data_ptr(), None)
    assert all(call(*a) != 0 for a in ((0, 64, 64), (1, 24, 64), (1, 64, 12), (1, 96, 96), (1, 528, 64), (1, 64, 64, 129), (1, 0, 64)))


@pytest.mark.parametrize("n", [2000, 6000])
def test_few_pairs_in_model_and_training_take_float_rows(n, monkeypatch):
    """SubMConv3d in inference and both directions of its training ask for them where the rule says so."""
    import numpy as np

    from pointtransformerv3_amd import ops
    from pointtransformerv3_amd.sparse import SparseConvTensor, SubMConv3d
    grid, batch, _ = unique_voxels(np.random.default_rng(n), n, 30, nb=1)
    idx = to_dev(np.concatenate([batch[:, None], grid], 1).astype(np.int32))
    seen, real = [], ops.subm_conv_pairs
    monkeypatch.setattr(ops, "subm_conv_pairs", lambda *a, wide=False: seen.append(wide) or real(*a, wide=wide))
    conv = SubMConv3d(128, 128, 3, bias=True, indice_key="k").half().to(DEV)
    x = torch.randn(n, 128, device=DEV, dtype=torch.half, requires_grad=True)
    sparse = lambda: SparseConvTensor(x, idx, [128] * 3, 1)
    with torch.no_grad():
        conv(sparse())
    conv(sparse()).features.sum().backward()
    assert seen == [True] * 3
