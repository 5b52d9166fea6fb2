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
