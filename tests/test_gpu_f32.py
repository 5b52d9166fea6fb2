"""The fp32 matrix-core products: Linear layers and the pair form of the convolution, at tile edges and odd widths."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, rel_err, to_dev, unique_voxels
from oracle import functional as OF
from oracle import indexing as OI

pytestmark = pytest.mark.gpu


def ops():
    from pointtransformerv3_amd import ops as o
    return o


@pytest.mark.parametrize("n,k,nout", [(1, 32, 32), (63, 6, 32), (64, 16, 64), (65, 17, 65), (129, 64, 33), (1000, 130, 192),
                                      (40_000, 64, 256), (70_000, 32, 128), (20_000, 128, 512)])
@pytest.mark.parametrize("gelu,resid", [(False, False), (True, True)])
def test_linear_f32_matches_double(n, k, nout, gelu, resid):
    g = torch.Generator().manual_seed(n + k + nout)
    x, w, b = (torch.randn(*s, generator=g) for s in ((n, k), (nout, k), (nout,)))
    r = torch.randn(n, nout, generator=g) if resid else None
    want = torch.nn.functional.linear(x.double(), w.double(), b.double())
    want = torch.nn.functional.gelu(want) if gelu else want
    want = want + r.double() if resid else want
    got = ops().linear_any(x.to(DEV), w.to(DEV), b.to(DEV), gelu=gelu, resid=None if r is None else r.to(DEV))
    assert rel_err(got, want) < 2e-6


@pytest.mark.parametrize("n,k,nout", [(5, 64, 192), (2049, 512, 512)])
def test_linear_f32_halves_on_one_side(n, k, nout):
    g = torch.Generator().manual_seed(n)
    x, w, b = (torch.randn(*s, generator=g).to(DEV) for s in ((n, k), (nout, k), (nout,)))
    o = ops()
    # a half result is the float one rounded once; half rows are the same rows converted
    assert torch.equal(o.linear_f32(x, w, b, torch.float16), o.linear_f32(x, w, b).half())
    assert torch.equal(o.linear_f32(x.half(), w, b), o.linear_f32(x.half().float(), w, b))


@pytest.mark.parametrize("ks,cin,cout,n,extent", [(3, 32, 32, 400, 12), (3, 64, 64, 3000, 18), (3, 128, 128, 60, 5),
                                                  (3, 20, 36, 700, 10), (5, 6, 32, 900, 14), (5, 3, 5, 40, 6),
                                                  (3, 256, 256, 1500, 14)])
def test_subm_conv_pairs_f32(ks, cin, cout, n, extent):
    rng = np.random.default_rng(cin + n)
    g = torch.Generator().manual_seed(cin + n)
    grid, batch, _ = unique_voxels(rng, n, extent, 2)
    idx = np.concatenate([batch[:, None].astype(np.int32), grid], 1)
    nbr = OI.subm_kmap(idx, ks)
    feat = torch.randn(len(idx), cin, generator=g)
    w = torch.randn(cout, ks ** 3, cin, generator=g) / (ks ** 3 * cin) ** 0.5
    b = torch.randn(cout, generator=g) if ks == 3 else None
    want = OF.subm_conv(feat, nbr, w, b)
    o = ops()
    plan = o.conv_plan_direct(to_dev(idx), ks)
    got = o.subm_conv_pairs(feat.to(DEV), plan, w.to(DEV), None if b is None else b.to(DEV))
    assert rel_err(got, want) < 5e-6
